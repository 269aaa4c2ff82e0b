"""Codec decoder on the GPU (q3t_decode_codes, q3t_stream_next_audio) against the float64 CPU
oracle of the reference's decoder (oracle/codec.py), on the synthetic speech-tokenizer
checkpoint.  Frame counts 3 and 10 put its linears and 1x1 convolutions on both matrix-core GEMM
kernels (few and many rows); at 70 frames a query block of the pre-transformer attention has five
16-key tiles, so that one of its four waves works on two."""
import numpy as np
import pytest

from oracle import codec as C
from q3t import engine as E
from q3t import synth

pytestmark = pytest.mark.gpu

# fp32 pipeline (exact bf16 x fp32 products, fp32 sums) over ~45 layers vs float64; samples
# are ~0.3 in magnitude and clamped to [-1, 1]
WAVE_TOL = 2e-3


@pytest.fixture(scope="module")
def codec_case(models):
    model, d = models.get_with_text("tiny")
    eng = E.HipTtsEngine(d, E.EngineOptions(max_cache_steps=128))
    yield eng, C.CodecOracle(synth.codec_tensors(0))
    eng.close()


@pytest.mark.parametrize("frames", [3, 10, 70])
def test_decode_matches_oracle(codec_case, frames):
    eng, oracle = codec_case
    assert eng.has_codec and eng.info["samples_per_frame"] == C.SAMPLES_PER_FRAME
    codes = np.random.default_rng(frames).integers(0, 2048, (frames, 16)).astype(np.int32)
    print(f"[gpu] decode_codes frames={frames}", flush=True)
    got = eng.decode_codes(codes)
    ref = oracle.decode(codes)
    assert got.shape == ref.shape == (frames * C.SAMPLES_PER_FRAME,)
    err = float(np.abs(got - ref).max())
    print(f"decode {frames} frames: max err {err:.2e}, mean |x| {float(np.abs(ref).mean()):.3f}")
    assert err <= WAVE_TOL


@pytest.mark.parametrize("frames", [1, 2, 5, 8, 9, 16, 17, 25, 26])
def test_decode_at_block_edges(codec_case, frames):
    """The decoder convolutions' 64-row blocks at half, exactly one and a remainder of a block
    (32 rows a frame after the first transposed convolution), split over channels, with rows
    before time 0 in every block; the attention's 16-row tiles (16, 17); and the frames at which the
    residual units of 96 channels (8, 9) and of 192 (25, 26) go from 32- to 64-row blocks.  ~45 layers of
    fp32 sums of exact products end within 3.4e-6 of float64 (2-norm) on inputs of 6 to 240 frames; four
    times that is allowed."""
    eng, oracle = codec_case
    codes = np.random.default_rng(100 + frames).integers(0, 2048, (frames, 16)).astype(np.int32)
    print(f"[gpu] decode_codes frames={frames}", flush=True)
    got, ref = eng.decode_codes(codes), oracle.decode(codes)
    err = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
    print(f"decode {frames} frames: rel err {err:.2e}")
    assert err <= 1.4e-5


def test_decode_of_thousands_of_frames(codec_case, monkeypatch):
    """2,200 frames: the 96-channel units' 64-row blocks pass 65,535 in the 2,185th.  The last 12 frames
    against the oracle, whose convolutions run over the last 40 only: they and the upsampling stages
    look back less than 11 frames.  The bound is test_decode_at_block_edges's."""
    eng, oracle = codec_case

    def attention(q, k, v):  # causal_attention by heads, on BLAS
        mask = np.triu(np.ones((len(q), len(q)), dtype=bool), 1)
        out = np.empty_like(q)
        for h in range(q.shape[1]):
            s = np.ascontiguousarray(q[:, h]) @ np.ascontiguousarray(k[:, h].T) / np.sqrt(q.shape[2])
            s[mask] = -np.inf
            s = np.exp(s - s.max(axis=1, keepdims=True))
            out[:, h] = s @ np.ascontiguousarray(v[:, h]) / s.sum(axis=1, keepdims=True)
        return out

    rng = np.random.default_rng(2200)
    q, k, v = rng.standard_normal((3, 9, 2, 64))
    np.testing.assert_allclose(attention(q, k, v), C.causal_attention(q, k, v), rtol=1e-12, atol=1e-14)
    monkeypatch.setattr(C, "causal_attention", attention)
    codes = rng.integers(0, 2048, (2200, 16)).astype(np.int32)
    print("[gpu] decode_codes frames=2200", flush=True)
    got = eng.decode_codes(codes)
    assert got.shape == (2200 * C.SAMPLES_PER_FRAME,)
    t = oracle.t
    x = C.causal_conv(oracle.rvq(codes), t["decoder.pre_conv.conv.weight"], t["decoder.pre_conv.conv.bias"])
    x = oracle.pre_transformer(x)[-40:]
    ref = np.clip(oracle.decoder(oracle.upsample(oracle.upsample(x, 0), 1)), -1.0, 1.0)
    n = 12 * C.SAMPLES_PER_FRAME
    err = float(np.linalg.norm(got[-n:] - ref[-n:]) / np.linalg.norm(ref[-n:]))
    print(f"decode 2200 frames, last 12: rel err {err:.2e}")
    assert err <= 1.4e-5


# Where a Snake stands: on the initial convolution's output, a 7-tap convolution's input and output rows,
# the 1x1 convolution's, twice inside a fused residual unit and on a fused unit's output.
SNAKES = ["1.block.0", "1.block.4.act1", "1.block.4.act2", "2.block.0", "3.block.3.act1", "3.block.3.act2", "5"]


def _one_channel_decoder(snake):
    """Codec tensors whose decoder carries one channel, known exactly, through `snake` alone: weights 0 but for
    channel 0, one factor per phase of a transposed convolution, every Snake but this one adds nothing
    (beta = 80), this one sin(x)^2 / (e^-19 + 1e-9) at alpha = 0.  Factors are short enough for 24 bits: in
    front of `snake` x is the same in fp32 and float64, between 1 and 5.4e8."""
    bits = lambda v: synth.f32_to_bf16_bits(np.asarray(v, dtype=np.float32)).reshape(np.shape(v))
    t = dict(synth.codec_tensors(0))
    for name in [n for n in t if n.startswith("decoder.decoder.")]:
        t[name] = np.full_like(t[name], bits(80.0) if name.endswith("beta") else 0)

    def put(name, index, value):
        t[name][index] = bits(value)

    first = 1.0 if snake != "1.block.0" else 131.0 * 2 ** 22
    put("decoder.decoder.0.conv.bias", 0, first)
    steps = ([3.0, 57.0 * 2 ** 4, 57.0 * 2 ** 10, 2.0 ** 16, 71.0 * 2 ** 11, 147.0 * 2 ** 15, 181.0 * 2 ** 20, 129.0 * 2 ** 22],
             [1, 3 / 4, 5 / 8, 7 / 8, 11 / 16], [1, 3 / 4, 5 / 8, 7 / 8], [1, 5 / 8, 7 / 8])
    for b, f in enumerate(steps):
        put(f"decoder.decoder.{b + 1}.block.1.conv.weight", (0, 0, slice(0, len(f))), f if first == 1 or b else 1)
    t[f"decoder.decoder.{snake}.beta"][:] = bits(-19.0)
    if ".act" in snake:  # its unit passes the channel on: x + Snake(x)
        unit = "decoder.decoder." + snake.rsplit(".", 1)[0]
        put(unit + ".conv1.conv.weight", (0, 0, 6), 1)
        put(unit + ".conv2.conv.weight", (0, 0, 0), 1)
    put("decoder.decoder.6.conv.weight", (0, 0, 6), 2.0 ** -31)
    return t


@pytest.mark.parametrize("snake", SNAKES)
def test_snake_of_large_arguments(models, tmp_path, monkeypatch, snake):
    """A Snake on both sides of the fast sine's range (65,536) and far past it, alone in front of the samples.
    Bound: sin within 1.2e-7, so sin^2 within 2.4e-7, and the scale within 4 roundings, 2.4e-7, together below
    1e-6 of the scale; and at most 16 roundings of x on its way, of 2^-24 of the largest.  The bound does
    not pass sin^2 left out past 65,536, nor the fast form past it (both planted in the oracle)."""
    tensors = _one_channel_decoder(snake)
    codes = np.zeros((1, 16), np.int32)
    oracle, scale = C.CodecOracle(tensors), 2.0 ** -31 / (np.exp(-19.0) + 1e-9)
    ref = oracle.decode(codes)
    assert 0.1 < np.abs(ref).max() < 1
    bound = 1e-6 * scale + 16 * 2.0 ** -24 * np.abs(ref).max()

    def planted(sin2):
        def snake_form(x, log_alpha, log_beta):
            y = x * np.exp(log_alpha)
            return x + np.where(np.abs(y) < 65536, np.sin(y) ** 2, sin2(y)) / (np.exp(log_beta) + 1e-9)
        with monkeypatch.context() as m:
            m.setattr(C, "snake", snake_form)
            return np.abs(oracle.decode(codes) - ref).max()

    def fast(y):  # fp32: n = rint(y / pi), r = y - n pi with pi in two parts, a sine that holds to 1.62
        f = lambda v: v.astype(np.float32).astype(np.float64)
        n = np.rint(f(y * np.float64(np.float32(1 / np.pi))))
        hi = np.float64(np.float32(np.pi))
        r = f(f(y - n * hi) - n * np.float64(np.float32(np.pi - hi)))
        return np.where(np.abs(r) <= 1.62, np.sin(r) ** 2, 2.0)

    if snake == SNAKES[-1]:
        assert planted(np.sin) > 100 * bound and planted(np.zeros_like) > 100 * bound and planted(fast) > 100 * bound
    model, _ = models.get("tiny")
    model.write(str(tmp_path))
    synth.write_codec(str(tmp_path), 0, tensors)
    print(f"[gpu] decode_codes, large arguments of Snake {snake}", flush=True)
    with E.HipTtsEngine(str(tmp_path), E.EngineOptions(max_cache_steps=64)) as eng:
        got = eng.decode_codes(codes)
    err = float(np.abs(got - ref).max())
    print(f"Snake {snake}: max err {err:.2e} of {bound:.2e}")
    assert err <= bound


def test_decode_is_causal_and_wraps_codes(codec_case):
    eng, _ = codec_case
    codes = np.random.default_rng(7).integers(0, 2048, (8, 16)).astype(np.int32)
    full = eng.decode_codes(codes)
    head = eng.decode_codes(codes[:5])
    np.testing.assert_allclose(head, full[:5 * C.SAMPLES_PER_FRAME], rtol=0, atol=1e-5)
    wrapped = codes.copy()
    wrapped[:, 4] += 2048                      # codes are taken modulo the codebook size
    np.testing.assert_array_equal(eng.decode_codes(wrapped), full)
    assert eng.decode_codes(np.zeros((0, 16), np.int32)).size == 0


def test_stream_audio_chunks(codec_case):
    eng, oracle = codec_case
    from q3t.workloads import WORKLOADS
    w = WORKLOADS["tiny_greedy"]
    model, _ = eng, None
    inputs = w.inputs(synth.SyntheticModel.build("tiny", 0))
    opts = E.GenerateOptions.greedy(10)
    for ctx in (25, 2):
        st = eng.start_stream(inputs, opts, E.StreamOptions(left_context_frames=ctx))
        chunks = []
        while (c := st.next_audio_chunk(4)) is not None:
            assert c.samples.shape == (c.frames * C.SAMPLES_PER_FRAME,) and c.sample_rate == 24000
            chunks.append(c)
        codes = np.concatenate(st._codes)
        st.close()
        assert [c.frames for c in chunks] == [4, 4, 2]
        got = np.concatenate([c.samples for c in chunks])
        ref = np.concatenate([C.stream_chunk_samples(oracle, codes, s, e, ctx) for s, e in ((0, 4), (4, 8), (8, 10))])
        err = float(np.abs(got - ref).max())
        print(f"stream audio, left context {ctx}: max err {err:.2e}")
        assert err <= WAVE_TOL


def test_generate_returns_audio(codec_case):
    eng, _ = codec_case
    text = "hello world"
    sp = eng.generate(text, E.GenerateOptions.greedy(6, decode_audio=True))
    assert sp.frames == 6 and sp.samples.shape == (6 * C.SAMPLES_PER_FRAME,) and sp.sample_rate == 24000
    np.testing.assert_allclose(sp.samples, eng.decode_codes(sp.codes), rtol=0, atol=0)


def test_no_codec_checkpoint(models):
    _, plain = models.get("tiny")
    with E.HipTtsEngine(plain, E.EngineOptions(max_cache_steps=64)) as e2:
        assert not e2.has_codec
        with pytest.raises(E.NotFoundError):
            e2.decode_codes(np.zeros((2, 16), np.int32))
