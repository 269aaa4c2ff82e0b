"""The last bits of what the Talker's path returns: prompt rows, GEMMs of the batched frame and of
the prefill, and prefills, against digests recorded from this engine's first matrix-core kernels.

Every frame is an argmax or a draw over logits that depend on all sums before them.  Over a few
thousand frames some two logits are equal to a bit or two (sixteen streams of 64-240 frames come
across a margin of exactly zero), and a sum in another order, although no less accurate, then turns a
stream's codes from there on.  So the order of the additions is part of the result, and a kernel that
shares the work out in another way keeps it: K parts by shape (gemm_k_parts), one chain a part over
32-wide steps in low, middle, high terms, parts in order; attention tiles of 16 keys in order.

`python tests/test_gpu_sum_order.py FILE` writes the digests of the tree it is run in.
"""
import hashlib
import json
import os
import sys

import numpy as np
import pytest

if __name__ == "__main__":
    sys.path[:0] = [os.getcwd(), os.path.join(os.getcwd(), "qwen3-tts-hip_amd"), os.path.join(os.getcwd(), "tests")]

from q3t import engine as E
from q3t import synth, textprep

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "sum_order.json")

# The batched frame's GEMMs (up to 16 rows): plain, RMSNorm, residual, SwiGLU, K in two halves.
FRAME_GEMMS = [(1, 1024, 1024), (16, 1024, 1024), (7, 96, 512), (16, 208, 2048)]
# The prefill's, in one K part: the two kernels, whole and partial tiles, k steps that do not fill a wave's.
GEMMS = [(M, N, K) for M in (17, 33, 65, 129, 200) for N, K in ((192, 1024), (84, 96), (320, 160), (64, 3072))]
# Both projections, in 16 parts down to one: rows = ids + 11.
PROMPTS = [1, 5, 6, 21, 22, 53, 54, 85, 117, 118, 200, 300]
# Row counts at which a kernel, its share of the work or the number of parts changes.
PREFILLS = [("tiny", False, (1, 3, 16, 17, 40, 64, 65, 97, 128, 129, 193)), ("tiny", True, (5, 65, 130)),
            ("tiny-proj", False, (16, 33, 129)),
            ("0.6b", False, (9, 16, 17, 32, 41, 64, 65, 96, 129, 200, 257, 385, 521)), ("0.6b", True, (41, 300)),
            ("1.7b", False, (16, 30, 41, 65, 137))]


def digest(*arrays):
    h = hashlib.sha256()
    for a in arrays:
        h.update(np.ascontiguousarray(a).tobytes())
    return h.hexdigest()[:32]


def _operands(M, N, K):
    rng = np.random.default_rng([M, N, K])
    X = (rng.standard_normal((M, K)) * 2).astype(np.float32)
    W = synth.f32_to_bf16_bits((rng.standard_normal((2 * N, K)) * 0.05).astype(np.float32))
    return (X, W, (1 + 0.1 * rng.standard_normal(K)).astype(np.float32),
            rng.standard_normal((M, N)).astype(np.float32), rng.standard_normal(N).astype(np.float32))


def gemm_digest(eng, M, N, K):
    X, W, g, res, b = _operands(M, N, K)
    out = [eng.debug_gemm(0, X, W[:N], N), eng.debug_gemm(0, X, W[:N], N, gamma=g),
           eng.debug_gemm(1, X, W[:N], N, res=res), eng.debug_gemm(3, X, W[:N], N, bias=b)]
    if N % 16 == 0:
        out.append(eng.debug_gemm(2, X, W, N, gamma=g))
    if M <= 16 and K % 1024 == 0 and N % 32 == 0:
        out.append(eng.debug_gemm(4, X, W[:N], N, res=res))
    return digest(*out)


def prompt_digest(eng, n):
    p = eng.prepare_text(textprep.random_prompt(n, 40 + n))
    return digest(p.prefill, p.trailing_text, p.tts_pad_embed)


def prefill_digest(eng, hidden, P):
    x = (np.random.default_rng([hidden, P]).standard_normal((P, hidden)) * 0.1).astype(np.float32)
    h, logits, _ = eng.debug_talker_prefill(x)
    return digest(h, logits)


def _engine(models, spec, kv_bf16=False, text=False):
    model, d = (models.get_with_text if text else models.get)(spec)
    return model, E.HipTtsEngine(d, E.EngineOptions(max_cache_steps=640, kv_bf16=kv_bf16))


@pytest.fixture(scope="module")
def golden():
    with open(GOLDEN) as f:
        return json.load(f)


@pytest.fixture(scope="module")
def tiny(models):
    _, eng = _engine(models, "tiny")
    yield eng
    eng.close()


@pytest.mark.parametrize("M,N,K", FRAME_GEMMS)
def test_frame_gemm(tiny, golden, M, N, K):
    print(f"[gpu] sum order, frame gemm M={M} N={N} K={K}", flush=True)
    assert gemm_digest(tiny, M, N, K) == golden[f"gemm {M} {N} {K}"]


@pytest.mark.parametrize("M,N,K", GEMMS)
def test_gemm(tiny, golden, M, N, K):
    print(f"[gpu] sum order, gemm M={M} N={N} K={K}", flush=True)
    assert gemm_digest(tiny, M, N, K) == golden[f"gemm {M} {N} {K}"]


@pytest.mark.parametrize("spec", ["tiny", "0.6b"])
def test_prompt_rows(models, golden, spec):
    _, eng = _engine(models, spec, text=True)
    with eng:
        for n in PROMPTS:
            print(f"[gpu] sum order, prompt {spec} ids={n}", flush=True)
            assert prompt_digest(eng, n) == golden[f"prompt {spec} {n}"], n


@pytest.mark.parametrize("spec,kv_bf16,rows", PREFILLS)
def test_prefill(models, golden, spec, kv_bf16, rows):
    model, eng = _engine(models, spec, kv_bf16)
    with eng:
        for P in rows:
            print(f"[gpu] sum order, prefill {spec} kv_bf16={kv_bf16} P={P}", flush=True)
            got = prefill_digest(eng, model.spec.talker.hidden, P)
            assert got == golden[f"prefill {spec} {kv_bf16} {P}"], P


if __name__ == "__main__":
    from conftest import _ModelCache

    cache, out = _ModelCache(), {}
    with _engine(cache, "tiny")[1] as eng:
        for M, N, K in FRAME_GEMMS + GEMMS:
            out[f"gemm {M} {N} {K}"] = gemm_digest(eng, M, N, K)
    for spec in ("tiny", "0.6b"):
        with _engine(cache, spec, text=True)[1] as eng:
            for n in PROMPTS:
                out[f"prompt {spec} {n}"] = prompt_digest(eng, n)
    for spec, kv_bf16, rows in PREFILLS:
        model, eng = _engine(cache, spec, kv_bf16)
        with eng:
            for P in rows:
                out[f"prefill {spec} {kv_bf16} {P}"] = prefill_digest(eng, model.spec.talker.hidden, P)
    with open(sys.argv[1], "w") as f:
        json.dump(out, f, indent=0, sort_keys=True)
        f.write("\n")
    cache.close()
