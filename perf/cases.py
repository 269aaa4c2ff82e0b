"""The calls a user of the engine makes, as measurable cases.

Six kinds of call, each through the Python mirror of the engine API (q3t.engine):

  prompt   HipTtsEngine.prepare_text: content token ids -> prompt rows
  prefill  HipTtsEngine.debug_talker_prefill: the Talker over the rows of a prompt -> hidden, logits, token
  audio    HipTtsEngine.decode_codes: codec frames -> 24 kHz samples
  first    start_stream + the first next_audio_chunk: what a listener waits for
  stream   start_stream + next_codes_chunk until the stream ends, the Talker's logits beside the codes
  serve    start_streams + next_codes_chunks over ragged streams, then every stream's audio

The shapes are the repository's own ("0.6b", "1.7b", random weights of seed 0, the synthetic codec),
the sizes those of q3t.workloads and bench.py and the ranges around them.  Weights and engines are what
a program loads once and keeps, so they are kept here too, one engine per set of engine options; prompts
and codes come from the seed.
"""
import json
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "qwen3-tts-hip_amd")  # run from the repository's root
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from q3t import engine as E  # noqa: E402
from q3t import synth  # noqa: E402

CONTENT_IDS = 151643  # content ids are below the special ones
CHUNK = 6             # frames of a streaming pull, as q3t.workloads pulls them


# ----------------------------------------------------------------------------------------
# the cases
# ----------------------------------------------------------------------------------------
def listed():
    return [
        # a short reply's prompt: the smallest call, bound by launches, copies and allocations
        dict(name="prompt_12", kind="prompt", spec="0.6b", ids=12),
        # a long paragraph's prompt at the wider model
        dict(name="prompt_487_1.7b", kind="prompt", spec="1.7b", ids=487),
        # the Talker over a one-sentence prompt (32 content tokens, all in the prefill)
        dict(name="prefill_41", kind="prefill", spec="0.6b", steps=41, kv_bf16=False),
        # the longest prompt of the multi-stream workload, with the bf16 KV cache
        dict(name="prefill_521_bf16kv", kind="prefill", spec="0.6b", steps=521, kv_bf16=True),
        # a 128-token prompt on the wider model, an odd number of rows
        dict(name="prefill_137_1.7b", kind="prefill", spec="1.7b", steps=137, kv_bf16=False),
        # the first window of a stream: six frames, no context yet
        dict(name="audio_6", kind="audio", frames=6),
        # every later window: a pull of 6 with 25 frames of left context
        dict(name="audio_31", kind="audio", frames=31),
        # a whole utterance (19.2 s) decoded at once
        dict(name="audio_240", kind="audio", frames=240),
        # time to first audio: prompt rows, 16-row prefill, six frames and their samples
        dict(name="first_audio", kind="first", ids=64, lookahead=7),
        # one greedy stream, 240 frames in pulls of six at a capacity of 256 (the headline setting)
        dict(name="stream_greedy", kind="stream", spec="0.6b", ids=64, lookahead=7, frames=240, cap=256, sample=False),
        # the same with the default sampling options on both heads, a shorter utterance
        dict(name="stream_sampled", kind="stream", spec="0.6b", ids=33, lookahead=8, frames=97, cap=256, sample=True),
        # sixteen listeners: prompts of 16-512 tokens, 64-240 frames each
        dict(name="serve_16", kind="serve", streams=16, ids_min=16, ids_max=512, frames_min=64, frames_max=240,
             sampled_every=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))


def draw(rng):
    kind = rng.choice(["prompt", "prefill", "prefill", "audio", "audio", "first", "stream", "stream", "serve"])
    if kind == "prompt":
        return dict(kind=kind, spec=rng.choice(["0.6b", "1.7b"]), ids=_log(rng, 1, 512))
    if kind == "prefill":
        return dict(kind=kind, spec=rng.choice(["0.6b", "0.6b", "1.7b"]), steps=_log(rng, 10, 521),
                    kv_bf16=rng.random() < 0.3)
    if kind == "audio":
        return dict(kind=kind, frames=_log(rng, 1, 240))
    if kind == "first":
        return dict(kind=kind, ids=_log(rng, 2, 200), lookahead=rng.randint(1, 7))
    if kind == "stream":
        spec = rng.choice(["0.6b", "0.6b", "1.7b"])
        return dict(kind=kind, spec=spec, ids=_log(rng, 4, 160), lookahead=rng.randint(1, 12), frames=_log(rng, 6, 140),
                    cap=256 if spec == "0.6b" else 512, sample=rng.random() < 0.4)
    # options mixed among the streams of a batch, as independent listeners choose them
    return dict(kind=kind, streams=rng.randint(2, 16), ids_min=4, ids_max=320, frames_min=8, frames_max=72,
                sampled_every=rng.choice([0, 0, 2, 3]))


# ----------------------------------------------------------------------------------------
# models, engines, inputs
# ----------------------------------------------------------------------------------------
_engines = {}
MODELS = os.path.join(tempfile.gettempdir(), f"q3t_perf_models_{os.getuid()}")


def _model_dir(spec):
    """The checkpoint of `spec` (with text table and codec), written once per machine."""
    d = os.path.join(MODELS, spec)
    if not os.path.exists(os.path.join(d, "complete")):
        synth.SyntheticModel.build(spec, 0).write(d, text_embedding=True)
        synth.write_codec(d, 0)
        with open(os.path.join(d, "complete"), "w") as f:
            f.write("ok\n")
    return d


def _engine(spec, cap=256, streams=1, kv_bf16=False, trace=False):
    key = (spec, cap, streams, kv_bf16, trace)
    if key not in _engines:
        eng = E.HipTtsEngine(_model_dir(spec), E.EngineOptions(device=0, max_cache_steps=cap, max_streams=streams,
                                                              kv_bf16=kv_bf16))
        if trace:
            eng.set_trace(True)
        _engines[key] = eng
    return _engines[key]


def _case_engine(case):
    k = case["kind"]
    if k == "prefill":
        return _engine(case["spec"], 768, kv_bf16=case["kv_bf16"])
    if k == "stream":
        return _engine(case["spec"], case["cap"], trace=True)
    if k == "serve":
        return _engine("0.6b", 768, streams=16)
    return _engine(case.get("spec", "0.6b"))


def _rng(case, seed):
    text = json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True)
    return np.random.default_rng([seed, *text.encode()])


def _ids(rng, n):
    return [int(i) for i in rng.integers(0, CONTENT_IDS, n)]


def _options(frames, sample, seed):
    if sample:  # the defaults of GenerateOptions
        return E.GenerateOptions(max_frames=frames, decode_audio=False, seed=seed)
    return E.GenerateOptions.greedy(frames)


def _plan(case):
    """Every stream's prompt length and frames: part of the case, not of its inputs."""
    n, rng = case["streams"], _rng(case, 0)
    lengths = rng.integers(case["ids_min"], case["ids_max"] + 1, n)
    frames = rng.integers(case["frames_min"], case["frames_max"] + 1, n)
    return [int(x) for x in lengths], [int(x) for x in frames]


def _prefill_rows(case, seed):
    # prompt rows are sums of a projected text embedding and a codec embedding row, N(0, 0.02) each
    H = synth.SPECS[case["spec"]].talker_hidden
    return (_rng(case, seed).standard_normal((case["steps"], H)) * 0.028).astype(np.float32)


def _codes(case, seed):
    return _rng(case, seed).integers(0, 2048, (case["frames"], 16)).astype(np.int32)


def prepare(case, seed):
    rng = _rng(case, seed)
    st = dict(case=case, eng=_case_engine(case))
    k = case["kind"]
    if k in ("prompt", "first", "stream"):
        st["ids"] = _ids(rng, case["ids"])
    if k == "prefill":
        st["rows"] = _prefill_rows(case, seed)
    elif k == "audio":
        st["codes"] = _codes(case, seed)
    elif k == "first":
        st["options"] = _options(240, False, seed)
        st["stream_options"] = E.StreamOptions(text_lookahead_tokens=case["lookahead"])
    elif k == "stream":
        st["options"] = _options(case["frames"], case["sample"], seed)
        st["stream_options"] = E.StreamOptions(text_lookahead_tokens=case["lookahead"])
    elif k == "serve":
        lengths, frames = _plan(case)
        every = case["sampled_every"]
        st["inputs"] = [_ids(rng, n) for n in lengths]
        st["options"] = [_options(f, bool(every) and j % every == every - 1, j) for j, f in enumerate(frames)]
        st["stream_options"] = E.StreamOptions(text_lookahead_tokens=1 << 30)
    return st


def _padded(a, n, fill):
    """a in an array of n rows: a stream may end before its last frame."""
    out = np.full((n,) + a.shape[1:], fill, a.dtype)
    out[:a.shape[0]] = a
    return out


def run(state):
    eng, k = state["eng"], state["case"]["kind"]
    if k == "prompt":
        p = eng.prepare_text(state["ids"])
        return dict(prefill=p.prefill, trailing=p.trailing_text, pad=p.tts_pad_embed)
    if k == "prefill":
        hidden, logits, token = eng.debug_talker_prefill(state["rows"])
        return dict(hidden=hidden, logits=logits, token=token)
    if k == "audio":
        return dict(samples=eng.decode_codes(state["codes"]))
    if k == "first":
        with eng.start_stream(state["ids"], state["options"], state["stream_options"]) as s:
            chunk = s.next_audio_chunk(CHUNK)
            return dict(samples=chunk.samples if chunk else np.zeros(0, np.float32),
                        codes=np.concatenate(s._codes) if s._codes else np.zeros((0, 16), np.int32))
    if k == "stream":
        with eng.start_stream(state["ids"], state["options"], state["stream_options"]) as s:
            parts = []
            while (c := s.next_codes_chunk(CHUNK)) is not None:
                parts.append(c.codes)
            codes = np.concatenate(parts) if parts else np.zeros((0, 16), np.int32)
            n = state["case"]["frames"]
            return dict(codes=_padded(codes, n, -1), logits=_padded(s.talker_logits(), n, 0.0))
    streams = eng.start_streams(state["inputs"], state["options"], state["stream_options"])
    try:
        live = list(streams)
        while live:
            chunks = eng.next_codes_chunks(live, CHUNK)
            live = [s for s, c in zip(live, chunks) if c is not None]
        codes = [s.finish_codes().codes for s in streams]
    finally:
        for s in streams:
            s.close()
    frames = [o.max_frames for o in state["options"]]
    return dict(codes=[_padded(c, n, -1) for c, n in zip(codes, frames)],
                samples=[_padded(eng.decode_codes(c), n * E.SAMPLES_PER_FRAME, 0.0) for c, n in zip(codes, frames)])


# ----------------------------------------------------------------------------------------
# the work a case cannot do without, and what its results may differ by
# ----------------------------------------------------------------------------------------
def _stack_params(s):
    q, kv = s.q_heads * s.head_dim, s.kv_heads * s.head_dim
    return s.layers * ((q + 2 * kv) * s.hidden + s.hidden * q + 3 * s.intermediate * s.hidden)


def _kv_bytes(s, elem=4):
    return s.layers * 2 * s.kv_heads * s.head_dim * elem


def _prompt_work(spec, ids):
    s = synth.SPECS[spec]
    rows = ids + 11
    w = s.text_hidden * s.text_proj_intermediate + s.text_proj_intermediate * s.talker_hidden
    return 2 * w + rows * (2 * s.text_hidden + 4 * s.talker_hidden), 2 * w * rows


def _prefill_work(spec, steps, kv=4):
    t = synth.SPECS[spec].talker
    w = _stack_params(t)
    attn = t.layers * 2 * t.q_heads * t.head_dim * steps * (steps + 1)
    return (2 * (w + t.vocab * t.hidden) + steps * (4 * t.hidden + _kv_bytes(t, kv)),
            2 * w * steps + 2 * t.vocab * t.hidden + attn)


def _codec_macs(frames):
    """Multiply-adds of the codec decoder per call, from its layer shapes."""
    c = synth.CODEC
    m = 2 * c["codebook_dim"] * c["projected"] + 3 * c["projected"] * c["pre_conv"]
    q = c["heads"] * c["head_dim"]
    m += 2 * c["pre_conv"] * c["hidden"] + c["layers"] * (4 * q * c["hidden"] + 3 * c["hidden"] * c["intermediate"])
    t = 1
    for _ in range(2):
        m += t * 2 * c["upsample"] ** 2
        t *= 2
        m += t * 2 * c["upsample"] * c["convnext"]
    m += t * 7 * c["upsample"] * c["decoder_init"]
    for ci, co, s in c["blocks"]:
        m += t * 2 * s * ci * co
        t *= s
        m += t * 3 * 8 * co * co
    return frames * (m + t * 7 * c["final"])


def _codec_work(frames):
    weights = sum(2 * int(np.prod(shape)) for name, shape, _ in synth.codec_inventory() if "_codebook" not in name)
    return weights + frames * (64 + 16 * 256 * 4 + 1920 * 4), 2 * _codec_macs(frames)


def _frame_work(spec, position, rows=1):
    """One frame of `rows` streams: the Talker's weights once, the CodePredictor's once per group
    (each group's input is the token of the one before), every cached row of every stream."""
    s = synth.SPECS[spec]
    t, c = s.talker, s.code_predictor
    wt, wc = _stack_params(t) + t.vocab * t.hidden, _stack_params(c) + c.vocab * c.hidden
    groups = s.num_code_groups - 1
    if s.has_projection:
        wc += t.hidden * c.hidden
    b = 2 * (wt + groups * wc) + rows * _kv_bytes(t) * position
    return b, 2 * rows * (wt + (groups + 1) * wc)


def _rollout_work(spec, ids, lookahead, frames):
    b, f = _prompt_work(spec, ids)
    p = 9 + max(1, min(lookahead, ids))
    b2, f2 = _prefill_work(spec, p)
    b3, f3 = _frame_work(spec, p + frames / 2)
    return b + b2 + frames * b3, f + f2 + frames * f3


def work(case):
    k = case["kind"]
    if k == "prompt":
        b, f = _prompt_work(case["spec"], case["ids"])
    elif k == "prefill":
        b, f = _prefill_work(case["spec"], case["steps"], 2 if case["kv_bf16"] else 4)
    elif k == "audio":
        b, f = _codec_work(case["frames"])
    elif k == "first":
        b, f = _rollout_work("0.6b", case["ids"], case["lookahead"], CHUNK)
        b2, f2 = _codec_work(CHUNK)
        b, f = b + b2, f + f2
    elif k == "stream":
        b, f = _rollout_work(case["spec"], case["ids"], case["lookahead"], case["frames"])
    else:
        lengths, frames = _plan(case)
        rows = sum(9 + n for n in lengths)
        b, f = _prefill_work("0.6b", rows)
        for i in range(max(frames)):
            live = [9 + n + i for n, fr in zip(lengths, frames) if fr > i]
            b1, f1 = _frame_work("0.6b", sum(live) / len(live), len(live))
            b, f = b + b1, f + f1
        b2, f2 = _codec_work(sum(frames))
        b, f = b + b2, f + f2
    return dict(bytes=float(b), flops=float(f))


def tolerance(case):
    """About four times the error seen against exact(), relative to the 2-norm of the result."""
    k = case["kind"]
    # exact products, fp32 sums over K <= 2048, two layers (seen: 1.4e-7)
    if k == "prompt":
        return {"rel": 6e-7}
    # 28 layers of fp32 sums (seen: 6e-7, and 3.8e-6 on the wider model); a bf16 KV cache rounds each K
    # and V value once, and a sum that ends a last bit apart rounds some of them to the next bf16 (seen: 6.5e-4)
    if k == "prefill":
        return {"rel": 2.6e-3 if case["kv_bf16"] else (1.6e-5 if case["spec"] == "1.7b" else 5e-6)}
    # ~45 layers of fp32 sums, twenty-nine sin^2 activations deep (seen: 3.4e-6)
    if k == "audio":
        return {"rel": 1.4e-5}
    # Tokens are argmaxes (or draws) over logits equal to ~1e-6, so they are the same but for a near tie,
    # which a few frames out of thousands come to; then the audio and the logits as above
    if k == "stream":
        return {"rel": 2e-5, "differ": 0.0}
    return {"rel": 1.4e-5, "differ": 0.0}


# ----------------------------------------------------------------------------------------
# 64-bit results in plain torch, from the checkpoint files
# ----------------------------------------------------------------------------------------
class _Weights:
    """float64 tensors of a BF16 safetensors file, read as they are asked for."""

    def __init__(self, path):
        with open(path, "rb") as f:
            n = struct.unpack("<Q", f.read(8))[0]
            self.head = json.loads(f.read(n))
        self.data = np.memmap(path, dtype=np.uint8, mode="r", offset=8 + n)

    def raw(self, name):
        m = self.head[name]
        b, e = m["data_offsets"]
        return self.data[b:e].view(np.int16).reshape(m["shape"])

    def __call__(self, name, rows=None):
        a = self.raw(name)
        a = np.ascontiguousarray(a if rows is None else a[rows])
        return torch.from_numpy(a).cuda().view(torch.bfloat16).double()


def _rms(x, g, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * g


def _rope(x, theta):
    T, _, d = x.shape
    inv = theta ** (-torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d)
    ang = torch.arange(T, dtype=torch.float64, device=x.device)[:, None] * inv
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, k, v):
    T, h, d = q.shape
    g = h // k.shape[1]
    out = torch.empty_like(q)
    mask = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1)
    for i in range(h):
        s = (q[:, i] @ k[:, i // g].T) / math.sqrt(d)
        out[:, i] = s.masked_fill(mask, -math.inf).softmax(-1) @ v[:, i // g]
    return out.reshape(T, h * d)


def _exact_prompt(case, seed):
    w = _Weights(os.path.join(_model_dir(case["spec"]), "model.safetensors"))
    ids = _ids(_rng(case, seed), case["ids"])
    tk = synth.TOKENS
    pad = tk["tts_pad_token_id"]
    spk, lang = synth.SPEAKER_IDS["ryan"], synth.LANGUAGE_IDS["english"]
    text = [tk["im_start_token_id"], tk["assistant_token_id"], 198] + [pad] * 5 + [tk["tts_bos_token_id"]] + ids
    codec = [None] * 3 + [tk["codec_think_id"], tk["codec_think_bos_id"], lang, tk["codec_think_eos_id"], spk,
                          tk["codec_pad_id"]] + [tk["codec_pad_id"]] * (len(ids) - 1) + [tk["codec_bos_id"]]
    text += [tk["tts_eos_token_id"], pad]
    x = w("talker.model.text_embedding.weight", text)
    p = "talker.text_projection.linear_fc"
    h = torch.nn.functional.silu(x @ w(p + "1.weight").T + w(p + "1.bias"))
    y = h @ w(p + "2.weight").T + w(p + "2.bias")
    emb = w("talker.model.codec_embedding.weight")
    for i, c in enumerate(codec):
        if c is not None:
            y[i] += emb[c]
    n = len(codec)
    return dict(prefill=y[:n], trailing=y[n:n + 1], pad=y[n + 1])


def _exact_prefill(case, seed):
    w = _Weights(os.path.join(_model_dir(case["spec"]), "model.safetensors"))
    t = synth.SPECS[case["spec"]].talker
    x = torch.from_numpy(_prefill_rows(case, seed)).cuda().double()
    T = x.shape[0]
    cache = (lambda a: a.float().bfloat16().double()) if case["kv_bf16"] else (lambda a: a)
    for i in range(t.layers):
        p = f"talker.model.layers.{i}."
        n = _rms(x, w(p + "input_layernorm.weight"), t.rms_eps)
        proj = lambda m: n @ w(p + f"self_attn.{m}_proj.weight").T
        q = _rms(proj("q").reshape(T, t.q_heads, t.head_dim), w(p + "self_attn.q_norm.weight"), t.rms_eps)
        k = _rms(proj("k").reshape(T, t.kv_heads, t.head_dim), w(p + "self_attn.k_norm.weight"), t.rms_eps)
        v = proj("v").reshape(T, t.kv_heads, t.head_dim)
        o = _attend(_rope(q, t.rope_theta), cache(_rope(k, t.rope_theta)), cache(v))
        x = x + o @ w(p + "self_attn.o_proj.weight").T
        n = _rms(x, w(p + "post_attention_layernorm.weight"), t.rms_eps)
        g = torch.nn.functional.silu(n @ w(p + "mlp.gate_proj.weight").T) * (n @ w(p + "mlp.up_proj.weight").T)
        x = x + g @ w(p + "mlp.down_proj.weight").T
    hidden = _rms(x[-1], w("talker.model.norm.weight"), t.rms_eps)
    logits = w("talker.codec_head.weight") @ hidden
    allowed = logits.clone()
    eos = allowed[synth.TOKENS["codec_eos_token_id"]].clone()
    allowed[t.vocab - 1024:] = -math.inf  # the last 1024 codec ids are specials; of them only eos is drawn
    allowed[synth.TOKENS["codec_eos_token_id"]] = eos
    return dict(hidden=hidden, logits=logits, token=int(allowed.argmax()))


def _conv(x, w, b, dilation=1):
    """Causal convolution over time-major rows: w [out, in, taps]."""
    T, k = x.shape[0], w.shape[2]
    xp = torch.cat([x.new_zeros((k - 1) * dilation, x.shape[1]), x])
    y = b.expand(T, -1).clone()
    for j in range(k):
        y += xp[j * dilation:j * dilation + T] @ w[:, :, j].T.contiguous()
    return y


def _up_conv(x, w, b, stride):
    """Transposed convolution, outputs past T * stride dropped: w [in, out, taps]."""
    T, k = x.shape[0], w.shape[2]
    y = x.new_zeros(T * stride + k, w.shape[1])
    for j in range(k):
        y[j:j + T * stride:stride] += x @ w[:, :, j].contiguous()
    return y[:T * stride] + b


def _exact_audio(case, seed):
    w = _Weights(os.path.join(_model_dir("0.6b"), "speech_tokenizer", "model.safetensors"))
    codes = torch.from_numpy(_codes(case, seed).astype(np.int64)).cuda()
    T = codes.shape[0]

    def book(p):
        return w(p + "._codebook.embedding_sum") / w(p + "._codebook.cluster_usage").clamp_min(1e-7)[:, None]

    def snake(x, p):
        return x + torch.sin(x * w(p + "alpha").exp()) ** 2 / (w(p + "beta").exp() + 1e-9)

    q = "decoder.quantizer.rvq_"
    rest = sum(book(f"{q}rest.vq.layers.{g}")[codes[:, g + 1]] for g in range(15))
    x = (book(q + "first.vq.layers.0")[codes[:, 0]] @ w(q + "first.output_proj.weight")[:, :, 0].T
         + rest @ w(q + "rest.output_proj.weight")[:, :, 0].T)
    x = _conv(x, w("decoder.pre_conv.conv.weight"), w("decoder.pre_conv.conv.bias"))
    t = "decoder.pre_transformer."
    h = x @ w(t + "input_proj.weight").T + w(t + "input_proj.bias")
    for i in range(8):
        p = f"{t}layers.{i}."
        n = _rms(h, w(p + "input_layernorm.weight"), 1e-5)
        q, k, v = ((n @ w(p + f"self_attn.{m}_proj.weight").T).reshape(T, 16, 64) for m in "qkv")
        o = _attend(_rope(q, 1e4), _rope(k, 1e4), v) @ w(p + "self_attn.o_proj.weight").T
        h = h + o * w(p + "self_attn_layer_scale.scale")
        n = _rms(h, w(p + "post_attention_layernorm.weight"), 1e-5)
        m = torch.nn.functional.silu(n @ w(p + "mlp.gate_proj.weight").T) * (n @ w(p + "mlp.up_proj.weight").T)
        h = h + m @ w(p + "mlp.down_proj.weight").T * w(p + "mlp_layer_scale.scale")
    x = _rms(h, w(t + "norm.weight"), 1e-5) @ w(t + "output_proj.weight").T + w(t + "output_proj.bias")
    for i in range(2):
        p = f"decoder.upsample.{i}."
        y = _up_conv(x, w(p + "0.conv.weight"), w(p + "0.conv.bias"), 2)
        p += "1."
        taps = w(p + "dwconv.conv.weight")[:, 0]
        yp = torch.cat([y.new_zeros(6, y.shape[1]), y])
        d = w(p + "dwconv.conv.bias") + sum(yp[j:j + y.shape[0]] * taps[:, j] for j in range(7))
        n = torch.nn.functional.layer_norm(d, d.shape[1:], w(p + "norm.weight"), w(p + "norm.bias"), 1e-6)
        a = torch.nn.functional.gelu(n @ w(p + "pwconv1.weight").T + w(p + "pwconv1.bias"))
        x = y + (a @ w(p + "pwconv2.weight").T + w(p + "pwconv2.bias")) * w(p + "gamma")
    d = "decoder.decoder."
    x = _conv(x, w(d + "0.conv.weight"), w(d + "0.conv.bias"))
    for b, (_, _, stride) in enumerate(synth.CODEC["blocks"]):
        p = f"{d}{b + 1}.block."
        x = _up_conv(snake(x, p + "0."), w(p + "1.conv.weight"), w(p + "1.conv.bias"), stride)
        for u, dil in enumerate((1, 3, 9)):
            r = f"{p}{u + 2}."
            a = _conv(snake(x, r + "act1."), w(r + "conv1.conv.weight"), w(r + "conv1.conv.bias"), dil)
            x = x + _conv(snake(a, r + "act2."), w(r + "conv2.conv.weight"), w(r + "conv2.conv.bias"))
    x = _conv(snake(x, d + "5."), w(d + "6.conv.weight"), w(d + "6.conv.bias"))
    return dict(samples=x[:, 0].clamp(-1.0, 1.0))


def exact(case, seed):
    if case["kind"] == "prompt":
        return _exact_prompt(case, seed)
    if case["kind"] == "prefill":
        return _exact_prefill(case, seed)
    if case["kind"] == "audio":
        return _exact_audio(case, seed)
    return None  # tokens feed back into what is computed: no such value
