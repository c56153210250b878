"""Performance cases of the decode path: the calls a text-to-speech program
makes, through the package's public entry points.

One utterance is: a prompt (a few rows for a built-in speaker, or hundreds of
rows of reference text and codes when a voice is cloned, or a kept voice
prefix plus the rows of the next text chunk), the frame loop, and the speech
decoder over the frames' codes.  Around it, programs that hold Q4 weights of
their own call the linear maps.  The weights are one synthetic checkpoint of
the 1.7B shapes (28-layer talker, 5-layer predictor, the 12 Hz speech
decoder), the same for every seed as a program's checkpoint is; the inputs
come from the seed.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qora-tts-12hz-1.7b_amd"))

import qtts  # noqa: E402
from qtts import synth  # noqa: E402

HIDDEN, VOCAB, INTER, LAYERS, HEADS, KV_HEADS, HEAD_DIM = 2048, 3072, 6144, 28, 16, 8, 128
TEXT_VOCAB = 151936
LANGUAGE, SPEAKER = 2055, 3000
KV_CAPACITY = 4096
TRAILING = 24                # text tokens still to be spoken, one per frame

# Linear maps of the checkpoint (talker and predictor, fused as they run) and
# two that no model holds, with ragged widths.
SHAPES = [(1024, 2048), (2048, 1024), (2048, 2048), (1024, 4096), (3072, 1024), (2048, 3072), (1024, 6144),
          (2048, 4096), (2048, 6144), (6144, 2048), (2048, 12288), (1000, 1500), (2080, 3000)]


def listed():
    return [
        # one row through a small map: a predictor head
        {"name": "gemv_1024x2048", "kind": "gemv", "k": 1024, "n": 2048},
        # one row through a wide map: a talker gate or up projection
        {"name": "gemv_2048x6144", "kind": "gemv", "k": 2048, "n": 6144},
        # a handful of rows at once, host arrays: short prompts, small batches
        {"name": "gemm_7x2048x4096", "kind": "gemm", "rows": 7, "k": 2048, "n": 4096, "device": False},
        # a cloned voice's prompt through the talker's gate|up, rows resident
        {"name": "gemm_400x2048x12288", "kind": "gemm", "rows": 400, "k": 2048, "n": 12288, "device": True},
        # one talker step of a caller's own loop, late in an utterance
        {"name": "step_kv2048", "kind": "step", "kv": 2048},
        # the frame loop late in an utterance, as a streaming program takes it
        {"name": "frames_16_kv2048", "kind": "frames", "kv": 2048, "frames": 16},
        # the shortest prompt: a built-in speaker and the first text token
        {"name": "prompt_builtin", "kind": "prompt", "text": 24},
        # a cloned voice: reference text and codes, the whole prompt at once
        {"name": "icl_400", "kind": "icl", "ref": 60, "text": 45, "frames": 390},
        # the same with a long reference, past one block of prompt rows
        {"name": "icl_1100", "kind": "icl", "ref": 170, "text": 61, "frames": 1090},
        # the next chunk of a text on a kept voice prefix
        {"name": "suffix_331_on_69", "kind": "suffix", "prefix": 69, "rows": 331},
        # an utterance's audio at once
        {"name": "audio_160", "kind": "audio", "frames": 160, "warmup": 0},
        # a streamed chunk of audio with the frames before it as warm-up
        {"name": "audio_13_after_8", "kind": "audio", "frames": 13, "warmup": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemm", "gemm", "step", "frames", "prompt", "icl", "suffix", "audio"])
    if kind == "gemv":
        k, n = rng.choice(SHAPES)
        return {"kind": kind, "k": k, "n": n + rng.choice([0, 0, 7])}
    if kind == "gemm":
        k, n = rng.choice(SHAPES)
        return {"kind": kind, "rows": _log_int(rng, 2, 700), "k": k, "n": n, "device": rng.random() < 0.5}
    if kind == "step":
        return {"kind": kind, "kv": _log_int(rng, 8, 3000)}
    if kind == "frames":
        return {"kind": kind, "kv": _log_int(rng, 8, 3000), "frames": rng.randint(1, 16)}
    if kind == "prompt":
        return {"kind": kind, "text": _log_int(rng, 2, 120)}
    if kind == "icl":
        frames = _log_int(rng, 12, 1090)
        return {"kind": kind, "ref": max(3, frames // rng.randint(4, 8)), "text": rng.randint(3, 90), "frames": frames}
    if kind == "suffix":
        return {"kind": kind, "prefix": rng.randint(12, 300), "rows": _log_int(rng, 2, 500)}
    return {"kind": kind, "frames": _log_int(rng, 1, 160), "warmup": rng.choice([0, 0, 4, 8, 25])}


# ---------------------------------------------------------------------------
# the program's checkpoint and contexts
# ---------------------------------------------------------------------------

_checkpoint = []             # (talker, predictor, decoder), made once per process
_idle = []                   # contexts with the checkpoint uploaded that no state holds


def _weights():
    if not _checkpoint:
        _checkpoint.append((synth.make_talker(seed=1, n_layers=LAYERS), synth.make_predictor(seed=2),
                            synth.make_decoder(seed=7)))
    return _checkpoint[0]


class State:
    """What one running request holds: a context with the checkpoint, its
    inputs and handles.  The context goes back to the program's idle ones."""

    def __init__(self, case):
        self.case, self.ctx, self.weight, self.prefix = case, None, None, None
        if _idle:
            self.ctx = _idle.pop()
            return
        talker, predictor, decoder = _weights()
        self.ctx = qtts.Context(0, kv_capacity=KV_CAPACITY)
        self.ctx.upload_model(talker, predictor)
        self.ctx.upload_decoder(decoder)

    def __del__(self):
        if self.ctx is None:
            return
        if self.weight is not None:
            self.weight.free()
        if self.prefix is not None:
            self.ctx.kv_reset()
            self.prefix.free()
        _idle.append(self.ctx)


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


def _rows(rng, *shape, scale=1.0):
    return (scale * rng.standard_normal(shape)).astype(np.float32)


def _cache(rng, n):
    """K after its norm and RoPE has unit rows; V is raw."""
    g = torch.Generator(device=_dev()).manual_seed(int(rng.integers(1 << 40)))
    K, V = (torch.randn((LAYERS, n, KV_HEADS, HEAD_DIM), generator=g, device=_dev()) for _ in "KV")
    return K.cpu().numpy(), (4 * V).cpu().numpy()


def _inputs(case, seed):
    """The inputs of a case as host arrays."""
    rng, kind = _rng(seed), case["kind"]
    if kind in ("gemv", "gemm"):
        w = synth.q4_random(rng, case["k"], case["n"])
        shape = (case["k"],) if kind == "gemv" else (case["rows"], case["k"])
        return {"w": w, "x": _rows(rng, *shape)}
    if kind == "step":
        return dict(zip("KV", _cache(rng, case["kv"])), x=_rows(rng, HIDDEN, scale=0.5))
    if kind == "frames":
        return dict(zip("KV", _cache(rng, case["kv"])), logits=_rows(rng, VOCAB, scale=4.0), hidden=_rows(rng, HIDDEN),
                    text=_rows(rng, TRAILING, HIDDEN, scale=0.5), pad=_rows(rng, HIDDEN, scale=0.5), seed=seed)
    if kind == "prompt":
        return {"text": rng.integers(0, 151000, case["text"]).astype(np.uint32)}
    if kind == "icl":
        return {"ref": rng.integers(0, 151000, case["ref"]).astype(np.uint32),
                "text": rng.integers(0, 151000, case["text"]).astype(np.uint32),
                "codes": rng.integers(0, 2048, (16, case["frames"])).astype(np.uint32),
                "voice": _rows(rng, HIDDEN, scale=0.5)}
    if kind == "suffix":
        return dict(zip("KV", _cache(rng, case["prefix"])), x=_rows(rng, case["rows"], HIDDEN, scale=0.5))
    return {"codes": rng.integers(0, 2048, (16, case["frames"])).astype(np.uint32),
            "warmup": rng.integers(0, 2048, (16, case["warmup"])).astype(np.uint32) if case["warmup"] else None}


def prepare(case, seed):
    s = State(case)
    s.inputs = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        s.weight = s.ctx.upload(s.inputs["w"])
        if case.get("device"):
            s.x = torch.from_numpy(s.inputs["x"]).cuda()
            s.y = torch.empty((case["rows"], case["n"]), dtype=torch.float32, device="cuda")
    elif kind in ("step", "frames", "suffix"):
        s.ctx.kv_load(s.inputs.pop("K"), s.inputs.pop("V"))
        if kind == "suffix":
            s.prefix = s.ctx.prefix_capture()
        if kind == "frames":
            s.params = qtts.sample_params(eos_enabled=False)
            s.ctx.gen_set_text(s.inputs["text"], s.inputs["pad"])
    return s


def run(s):
    case, ctx, i = s.case, s.ctx, s.inputs
    kind = case["kind"]
    if kind == "gemv":
        return ctx.gemv(s.weight, i["x"])
    if kind == "gemm":
        if not case["device"]:
            return ctx.gemm(s.weight, i["x"])
        ctx.gemm_noalloc(s.weight, s.x.data_ptr(), case["rows"], s.y.data_ptr())
        return s.y
    if kind == "step":
        ctx.kv_truncate(case["kv"])
        return ctx.forward_with_embedding(i["x"], case["kv"])
    if kind == "frames":
        ctx.kv_truncate(case["kv"])
        ctx.gen_begin(i["logits"], i["hidden"], case["kv"], i["seed"], s.params)
        codes, _ = ctx.gen_frames(case["frames"])
        logits, hidden, _, _ = ctx.gen_state()
        return {"codes": codes.astype(np.int64), "logits": logits, "hidden": hidden}
    if kind == "prompt":
        hidden, logits, _ = ctx.prefill_custom_voice(i["text"], SPEAKER, LANGUAGE)
        return {"hidden": hidden, "logits": logits, "trailing": ctx.build_trailing_text(i["text"])}
    if kind == "icl":
        rows, rest = ctx.build_icl_block(i["ref"], i["text"], i["codes"])
        hidden, logits, _ = ctx.prefill_custom_voice(i["text"], 0, LANGUAGE, i["voice"], rows)
        return {"rows": rows, "rest": rest, "hidden": hidden, "logits": logits}
    if kind == "suffix":
        ctx.prefix_attach(s.prefix)
        hidden = ctx.prefill_talker_raw_from(i["x"], case["prefix"])
        return {"hidden": hidden, "logits": ctx.apply_codec_head(hidden)}
    return ctx.decode_to_audio(i["codes"], i["warmup"])


# ---------------------------------------------------------------------------
# the least a pass has to move and compute
# ---------------------------------------------------------------------------

_LAYER = HIDDEN * 4096 + 2048 * HIDDEN + HIDDEN * 2 * INTER + INTER * HIDDEN      # weights of a talker layer
_PRED_LAYER = 1024 * 4096 + 2048 * 1024 + 1024 * 6144 + 3072 * 1024
_TEXT = 2 * HIDDEN * HIDDEN                                                       # the text projection
_KV_BYTES = 2 * KV_HEADS * HEAD_DIM * 4                                           # a cached position of one layer


def _q4(n):
    return 0.5625 * n


def _prefill(rows, start):
    """The talker over `rows` positions after `start` cached ones, and the
    codec head of the last."""
    attended = rows * start + rows * (rows + 1) / 2
    return (_q4(LAYERS * _LAYER + HIDDEN * VOCAB) + LAYERS * _KV_BYTES * (start + rows) + 4 * rows * HIDDEN
            + 4 * (HIDDEN + VOCAB),
            2 * (rows * LAYERS * _LAYER + HIDDEN * VOCAB) + LAYERS * 4 * HEADS * HEAD_DIM * attended)


def _audio(frames):
    d = _weights()[2]
    macs = weights = 0

    def conv(m, n, positions):
        nonlocal macs, weights
        macs, weights = macs + m * n * positions, weights + m * n

    t = frames
    conv(2 * d.codebook_dim, d.vq_dim, t)
    conv(d.vq_dim * d.pre_conv.kernel_size, d.latent, t)
    conv(d.latent, d.hidden, t)
    for _ in d.tf_layers:
        a = d.n_heads * d.head_dim
        conv(d.hidden, 3 * a, t)
        conv(a, d.hidden, t)
        conv(d.hidden, 3 * d.inter, t)
        macs += 2 * a * sum(min(j + 1, d.sliding_window) for j in range(t))
    conv(d.hidden, d.latent, t)
    for u in d.upsample:
        conv(d.latent * u.conv_t.kernel_size, d.latent, t)
        t *= u.conv_t.stride
        conv(7, d.latent, t)
        conv(d.latent, 2 * u.inner, t)
    conv(d.latent * 7, d.vocos_init.out_channels, t)
    for b in d.vocos_blocks:
        conv(b.upsample.in_channels * b.upsample.kernel_size, b.upsample.out_channels, t)
        t *= b.upsample.stride
        for r in b.residuals:
            conv(r.conv1.in_channels * 8, r.conv1.out_channels, t)
    conv(d.output_conv.in_channels * 7, 1, t)
    return 4 * weights + 4 * t + 64 * frames + 16 * 4 * d.codebook_dim * frames, 2 * macs


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        k, n, rows = case["k"], case["n"] // 32 * 32, case.get("rows", 1)
        return {"bytes": _q4(k * n) + 4 * rows * (k + case["n"]), "flops": 2 * rows * k * n}
    if kind == "step":
        b, f = _prefill(1, case["kv"])
        return {"bytes": b, "flops": f}
    if kind == "frames":
        b = f = 0
        for j in range(case["frames"]):
            tb, tf = _prefill(1, case["kv"] + j)
            pred = 16 * (5 * _PRED_LAYER + HIDDEN * 1024) + 15 * 1024 * 2048
            b, f = b + tb + _q4(5 * _PRED_LAYER + HIDDEN * 1024 + 15 * 1024 * 2048) + 64, f + tf + 2 * pred
        return {"bytes": b, "flops": f}
    if kind == "prompt":
        b, f = _prefill(10, 0)
        ids = case["text"] + 6
        return {"bytes": b + _q4(_TEXT) + ids * (0.5625 + 4) * HIDDEN, "flops": f + 2 * ids * _TEXT}
    if kind == "icl":
        rows = case["frames"] + 1
        b, f = _prefill(rows + 9, 0)
        ids = case["ref"] + case["text"] + 7
        return {"bytes": b + _q4(_TEXT) + rows * (16 * 0.5625 + 8) * HIDDEN, "flops": f + 2 * ids * _TEXT}
    if kind == "suffix":
        b, f = _prefill(case["rows"], case["prefix"])
        return {"bytes": b, "flops": f}
    b, f = _audio(case["frames"] + case["warmup"])
    return {"bytes": b, "flops": f}


def tolerance(case):
    """f32 arithmetic throughout (or a split that keeps its accuracy): the
    order of the sums is what differs, and how far that travels through the
    28 layers or the decoder's stages."""
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        return {"rel": 2e-6, "max": 2e-5}     # 2e-7 (one row) to 5e-7 off 64 bits
    if kind == "frames":
        # a tie within rounding picks another code, and every later one with it
        return {"rel": 3e-6, "max": 3e-5, "differ": 0.02}
    if kind == "audio":
        return {"rel": 3e-5, "max": 3e-4}     # 7.5e-6 off 64 bits
    return {"rel": 3e-6, "max": 3e-5}         # 1e-7 to 5e-7 off 64 bits


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------

def _t64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_dev()).double()


def _f16(a):
    return _t64(a.view(np.float16).astype(np.float32))


def _dense(w, rows=None):
    """A Q4 weight (or some of its rows) in 64 bits: low nibbles are the even
    columns, one scale per row and 32 columns, a partial group is zero."""
    packed, scales = (w.packed, w.scales) if rows is None else (w.packed[rows], w.scales[rows])
    p = torch.from_numpy(np.ascontiguousarray(packed)).to(_dev())
    k, g = p.shape[0], p.shape[1] // 16
    q = torch.stack([(p & 15).to(torch.int8), (p >> 4).to(torch.int8)], dim=-1).reshape(k, g, 32).double() - 8
    out = torch.zeros((k, w.n), dtype=torch.float64, device=q.device)
    out[:, : g * 32] = (q * _f16(scales).reshape(k, g, 1)).reshape(k, g * 32)
    return out


def _rms(x, gamma, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gamma


def _rope(x, cos, sin):
    """x [rows][heads][d], pairs (i, i + d/2)."""
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * cos[:, None] - b * sin[:, None], b * cos[:, None] + a * sin[:, None]], dim=-1)


def _silu(x):
    return x / (1 + torch.exp(-x))


def _talker(x, start, K=None, V=None):
    """The talker over rows x at positions start..: the last row's normed
    hidden and its codec logits."""
    t = _weights()[0]
    rows = x.shape[0]
    cos, sin = _t64(t.rope_cos[start:start + rows]), _t64(t.rope_sin[start:start + rows])
    pos = torch.arange(start + rows, device=x.device)
    hide = pos[None, :] > pos[start:, None]
    for j, L in enumerate(t.layers):
        h = _rms(x, _f16(L.input_norm))
        q = _rope(_rms((h @ _dense(L.q_proj)).reshape(rows, HEADS, HEAD_DIM), _f16(L.q_norm)), cos, sin)
        k = _rope(_rms((h @ _dense(L.k_proj)).reshape(rows, KV_HEADS, HEAD_DIM), _f16(L.k_norm)), cos, sin)
        v = (h @ _dense(L.v_proj)).reshape(rows, KV_HEADS, HEAD_DIM)
        if K is not None:
            k, v = torch.cat([_t64(K[j]), k]), torch.cat([_t64(V[j]), v])
        att = torch.empty_like(q)
        for i in range(HEADS):
            s = (q[:, i] @ k[:, i // 2].T) / math.sqrt(HEAD_DIM)
            att[:, i] = torch.softmax(s.masked_fill(hide, -math.inf), dim=-1) @ v[:, i // 2]
        x = x + att.reshape(rows, -1) @ _dense(L.o_proj)
        h = _rms(x, _f16(L.post_attn_norm))
        x = x + (_silu(h @ _dense(L.gate_proj)) * (h @ _dense(L.up_proj))) @ _dense(L.down_proj)
    h = _rms(x[-1], _f16(t.final_norm))
    return h, h @ _dense(t.codec_head)


def _text(ids):
    t = _weights()[0]
    h = _dense(t.text_embedding, np.asarray(ids, np.int64)) @ _dense(t.text_fc1) + _t64(t.text_fc1_bias)
    return _silu(h) @ _dense(t.text_fc2) + _t64(t.text_fc2_bias)


def _codec(ids):
    return _dense(_weights()[0].codec_embedding, np.asarray(ids, np.int64))


def _head(voice=None):
    """The 9 rows every prompt begins with: role, language, speaker."""
    text = _text([151644, 77091, 198, 151671, 151672])
    code = _codec([2154, 2156, LANGUAGE, 2157, 2148 if voice is not None else SPEAKER, 2148])
    if voice is not None:
        code[4] = _t64(voice)
    return torch.cat([text[:3], code[:5] + text[3], code[5:] + text[4]])


def _conv1d(x, c):
    pad = (c.kernel_size - 1) * c.dilation
    xp = torch.nn.functional.pad(x, (pad, 0))
    w, n = _t64(c.weight), x.shape[1]
    out = _t64(c.bias)[:, None].expand(-1, n).clone()
    for k in range(c.kernel_size):
        out += w[:, :, k].contiguous() @ xp[:, k * c.dilation:k * c.dilation + n].contiguous()
    return out


def _convt(x, c):
    """Transposed convolution, cropped to stride * positions."""
    w, n = _t64(c.weight), x.shape[1]
    full = torch.zeros((c.out_channels, (n - 1) * c.stride + c.kernel_size), dtype=torch.float64, device=x.device)
    for k in range(c.kernel_size):
        full[:, k:k + (n - 1) * c.stride + 1:c.stride] += w[:, :, k].T.contiguous() @ x
    return full[:, :n * c.stride] + _t64(c.bias)[:, None]


def _snake(x, alpha, beta):
    return x + torch.exp(-_t64(beta))[:, None] * torch.sin(torch.exp(_t64(alpha))[:, None] * x) ** 2


def _decode(codes):
    d = _weights()[2]
    c = torch.from_numpy(codes.astype(np.int64)).to(_dev())
    rest = sum(_t64(b)[c[g + 1]] for g, b in enumerate(d.rest_codebooks))
    x = (_t64(d.first_codebook)[c[0]] @ _t64(d.first_output_proj) + rest @ _t64(d.rest_output_proj)).T.contiguous()
    x = _conv1d(x, d.pre_conv).T @ _t64(d.tf_input_w) + _t64(d.tf_input_b)
    n = x.shape[0]
    cos, sin = _t64(d.rope_cos[:n]), _t64(d.rope_sin[:n])
    pos = torch.arange(n, device=x.device)
    hide = (pos[None] > pos[:, None]) | (pos[None] <= pos[:, None] - d.sliding_window)
    for L in d.tf_layers:
        h = _rms(x, _t64(L.input_norm), 1e-5)
        q, k = (_rope((h @ _t64(w)).reshape(n, d.n_heads, -1), cos, sin) for w in (L.q_proj, L.k_proj))
        v = (h @ _t64(L.v_proj)).reshape(n, d.n_heads, -1)
        att = torch.empty_like(q)
        for i in range(d.n_heads):
            s = (q[:, i] @ k[:, i].T) / math.sqrt(d.head_dim)
            att[:, i] = torch.softmax(s.masked_fill(hide, -math.inf), dim=-1) @ v[:, i]
        x = x + (att.reshape(n, -1) @ _t64(L.o_proj)) * _t64(L.attn_scale)
        h = _rms(x, _t64(L.post_attn_norm), 1e-5)
        x = x + ((_silu(h @ _t64(L.gate_proj)) * (h @ _t64(L.up_proj))) @ _t64(L.down_proj)) * _t64(L.mlp_scale)
    x = (_rms(x, _t64(d.tf_norm), 1e-5) @ _t64(d.tf_output_w) + _t64(d.tf_output_b)).T.contiguous()
    for u in d.upsample:
        x = _convt(x, u.conv_t)
        n = x.shape[1]
        xp, w = torch.nn.functional.pad(x, (u.dw_conv.kernel_size - 1, 0)), _t64(u.dw_conv.weight)
        h = _t64(u.dw_conv.bias)[:, None] + sum(w[:, k:k + 1] * xp[:, k:k + n] for k in range(u.dw_conv.kernel_size))
        mean = h.mean(0, keepdim=True)
        h = (h - mean) / torch.sqrt(((h - mean) ** 2).mean(0, keepdim=True) + 1e-5)
        h = (h * _t64(u.norm_w)[:, None] + _t64(u.norm_b)[:, None]).T @ _t64(u.pw1_w) + _t64(u.pw1_b)
        h = 0.5 * h * (1 + torch.tanh(h * 0.7071067811865476))
        x = x + _t64(u.gamma)[:, None] * (h @ _t64(u.pw2_w) + _t64(u.pw2_b)).T
    x = _conv1d(x, d.vocos_init)
    for b in d.vocos_blocks:
        x = _convt(_snake(x, b.pre_snake_alpha, b.pre_snake_beta), b.upsample)
        for r in b.residuals:
            h = _conv1d(_snake(x, r.act1_alpha, r.act1_beta), r.conv1)
            x = x + _conv1d(_snake(h, r.act2_alpha, r.act2_beta), r.conv2)
    return _conv1d(_snake(x, d.final_snake_alpha, d.final_snake_beta), d.output_conv)[0].clamp(-1, 1)


def exact(case, seed):
    kind = case["kind"]
    i = _inputs(case, seed)
    if kind in ("gemv", "gemm"):
        return _t64(i["x"]) @ _dense(i["w"])
    if kind == "step":
        return torch.cat(_talker(_t64(i["x"])[None], case["kv"], i["K"], i["V"]))
    if kind == "frames":
        return None          # the codes drawn are part of what is computed
    if kind == "prompt":
        first = _text(i["text"][:1]) + _codec([2149])
        hidden, logits = _talker(torch.cat([_head(), first]), 0)
        return {"hidden": hidden, "logits": logits, "trailing": _text(np.append(i["text"][1:], 151673))}
    if kind == "icl":
        p = _weights()[1]
        n = case["frames"] + 1
        text = _text(np.concatenate([i["ref"], i["text"], [151673]]))
        code = _codec(i["codes"][0])
        for g, e in enumerate(p.codec_embeddings):
            code = code + _dense(e, i["codes"][g + 1].astype(np.int64))
        code = torch.cat([_codec([2149]), code])
        side = torch.cat([text[:n], _text([151671]).expand(max(0, n - text.shape[0]), -1)])
        rows = side + code
        hidden, logits = _talker(torch.cat([_head(i["voice"]), rows]), 0)
        return {"rows": rows, "rest": text[n:], "hidden": hidden, "logits": logits}
    if kind == "suffix":
        hidden, logits = _talker(_t64(i["x"]), case["prefix"], i["K"], i["V"])
        return {"hidden": hidden, "logits": logits}
    warm = case["warmup"]
    codes = i["codes"] if not warm else np.concatenate([i["warmup"], i["codes"]], axis=1)
    y = _decode(codes)
    return y[warm * y.shape[0] // codes.shape[1]:]
