"""Talker prompt prefill at prompt lengths around the attention's 16-row query blocks and
16-key tiles (1, 2, 15, 16, 17, 33, 130 and
cap - 1), through the q3t_debug_talker_prefill hook, against the float64 oracle's prefill
(decode.rs:1077-1298).  Both query-head groupings (two query heads per KV head and one) and
both KV cache types (the oracle rounds K and V to bf16 where the GPU stores bf16)."""
import numpy as np
import pytest

from q3t import engine as E
from q3t import synth
from oracle.model import Oracle

pytestmark = pytest.mark.gpu

CAP = 200
LENGTHS = (1, 2, 15, 16, 17, 33, 130, CAP - 1)


def _close(got, want, max_tol, mean_tol, what):
    d = np.abs(np.asarray(got, np.float64) - np.asarray(want, np.float64))
    print(f"  {what}: max {d.max():.2e} mean {d.mean():.2e}")
    assert d.max() <= max_tol and d.mean() <= mean_tol, f"{what}: max {d.max():.3g} mean {d.mean():.3g}"


@pytest.mark.parametrize("spec", ["tiny", "tiny-g1"])
@pytest.mark.parametrize("kv_bf16", [False, True])
def test_prefill_lengths_match_oracle(models, spec, kv_bf16):
    model, d = models.get(spec, 0)
    H = model.spec.talker.hidden
    rng = np.random.default_rng(11)
    print(f"[gpu] prefill lengths {spec} kv_bf16={kv_bf16}", flush=True)
    with E.HipTtsEngine(d, E.EngineOptions(max_cache_steps=CAP, kv_bf16=kv_bf16)) as eng:
        for P in LENGTHS:
            x = (rng.standard_normal((P, H)) * 0.5).astype(np.float32)
            hidden, logits, _ = eng.debug_talker_prefill(x)
            o = Oracle(model.tensors, model.config(), max_cache_steps=CAP, kv_bf16=kv_bf16)
            want = o.prefill(x.astype(np.float64))
            # fp32 KV: ~7e-7 measured; bf16 KV: cache values on either side of a bf16
            # rounding boundary, ~6e-5 measured
            tol = (2e-3, 2e-4) if kv_bf16 else (1e-5, 1e-6)
            _close(hidden, o.hidden, *tol, f"P={P} hidden")
            _close(logits, want, *tol, f"P={P} logits")


@pytest.mark.parametrize("kv_bf16", [False, True])
def test_prefill_tiles_per_wave(models, kv_bf16):
    """Lengths around the attention's rounds of four 16-key tiles, one scored by each of its waves: 48 / 49
    and 63 .. 65 rows (three, four and five tiles), 80 / 81 and 128 / 129."""
    model, d = models.get("tiny", 0)
    rng = np.random.default_rng(12)
    print(f"[gpu] prefill tiles per wave kv_bf16={kv_bf16}", flush=True)
    with E.HipTtsEngine(d, E.EngineOptions(max_cache_steps=CAP, kv_bf16=kv_bf16)) as eng:
        for P in (48, 49, 63, 64, 65, 80, 81, 128, 129):
            x = (rng.standard_normal((P, model.spec.talker.hidden)) * 0.5).astype(np.float32)
            hidden, logits, _ = eng.debug_talker_prefill(x)
            o = Oracle(model.tensors, model.config(), max_cache_steps=CAP, kv_bf16=kv_bf16)
            want = o.prefill(x.astype(np.float64))
            # the bounds of test_prefill_lengths_match_oracle
            tol = (2e-3, 2e-4) if kv_bf16 else (1e-5, 1e-6)
            _close(hidden, o.hidden, *tol, f"P={P} hidden")
            _close(logits, want, *tol, f"P={P} logits")


def test_prefill_split_sums_leave_no_trace(models):
    """The O and down projections add onto the rows that they read as the residual, in K parts: the same
    prompt before and after others, through either GEMM kernel, gives the same bits."""
    model, d = models.get("tiny", 0)
    rng = np.random.default_rng(13)
    xs = [(rng.standard_normal((P, model.spec.talker.hidden)) * 0.5).astype(np.float32) for P in (41, 64, 65, 3, 130)]
    print("[gpu] prefill split sums", flush=True)
    with E.HipTtsEngine(d, E.EngineOptions(max_cache_steps=CAP)) as eng:
        first = [eng.debug_talker_prefill(x) for x in xs]
        for x, (hidden, logits, token) in list(zip(xs, first))[::-1]:
            h, l, t = eng.debug_talker_prefill(x)
            np.testing.assert_array_equal(h, hidden)
            np.testing.assert_array_equal(l, logits)
            assert t == token


@pytest.mark.parametrize("P", [65, 96, 97, 1023, 1024, 1025])
def test_prefill_tiled_split_sums(models, P):
    """O and down in 32-row tiles at hidden 512: K parts in two groups of waves a block, of 64 and of 128
    columns; whole and partial last tiles, the same bits when run again."""
    model, d = models.get("tiny", 0)
    x = (np.random.default_rng(P).standard_normal((P, model.spec.talker.hidden)) * 0.5).astype(np.float32)
    print(f"[gpu] prefill tiled split sums P={P}", flush=True)
    with E.HipTtsEngine(d, E.EngineOptions(max_cache_steps=1040)) as eng:
        hidden, logits, _ = eng.debug_talker_prefill(x)
        again = eng.debug_talker_prefill(x)
    np.testing.assert_array_equal(again[0], hidden)
    np.testing.assert_array_equal(again[1], logits)
    o = Oracle(model.tensors, model.config(), max_cache_steps=1040)
    want = o.prefill(x.astype(np.float64))
    # the bounds of test_prefill_lengths_match_oracle
    _close(hidden, o.hidden, 1e-5, 1e-6, f"P={P} hidden")
    _close(logits, want, 1e-5, 1e-6, f"P={P} logits")
