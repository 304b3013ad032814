"""The batched prompt's launches that spread little work over the chip, against
the oracle's sequential loop: RoPE/KV by element groups, attention with the
keys spread over a workgroup's wavefronts, projections in uneven K parts.

Bounds: those of test_gpu_prefill.py (`_prompt_check`).
"""
import ctypes as C

import numpy as np
import pytest

from dotllm_amd import Q4_0, Q4_K, Q5_K, Q6_K, Q8_0, _lib, synth
from dotllm_amd.engine import InferenceEngine, LoadedModel
from oracle import oracle as O
from oracle_pair import KV_MARGIN, OraclePair
from test_gpu_prefill import (FP32_LEVEL, KV_MIN, _prompt_check, oracle_threads, random_blocks,  # noqa: F401
                              row_rel_err)

pytestmark = pytest.mark.gpu
PARTS_MAX = 512 * 128 * 128   # floats of a parts buffer


def host_fn(name, args, restype=C.c_int):
    """One of the library's own launch rules (host code, not part of the C ABI):
    the tests assert that their sizes take the path they are about."""
    f = getattr(_lib.lib(), f"_ZN6llmdot{len(name)}{name}E{args}")
    f.restype = restype
    f.argtypes = [{"i": C.c_int, "j": C.c_uint32, "l": C.c_int64}[a] for a in args]
    return f


def plan(t, m, n, k):
    """(tokens per tile, K parts) of a batched product (prefill_plan)."""
    v = host_fn("prefill_plan", "jiiil", C.c_int64)(t, m, n, k, PARTS_MAX)
    return v & 0xFFFFFFFF, v >> 32


@pytest.mark.parametrize("rot", [60, 24, 2])
def test_prefill_partial_rotation(hip, monkeypatch, rot):
    """Heads of 64 of which 60 (30 pairs: one per thread), 24 (12 pairs: 4 per
    thread beside unrotated elements) or 2 elements rotate."""
    real = synth.metadata

    def metadata(spec, *a, **k):
        return [(n, t, rot if n.endswith("rope.dimension_count") else v) for n, t, v in real(spec, *a, **k)]

    monkeypatch.setattr(synth, "metadata", metadata)
    img = synth.build_image("tiny", seed=1234, context=96)
    _prompt_check(hip, img, synth.prompt(32000, 40, seed=5), 96, True, [0, 3])


@pytest.mark.parametrize("n,split,kv_fp16", [(2, None, False), (17, None, True), (33, None, False), (49, 47, True),
                                             (300, 283, False), (300, 283, True)])
def test_prefill_attention_key_split(hip, oracle_threads, n, split, kv_fp16):  # noqa: F811
    """Heads of 96 (two layers of the Phi-3-mini shape): fewer keys than the
    wavefronts' steps, a last query block of one row, a chunk behind a cache."""
    spec = dict(synth.SPECS["phi3mini"], layers=2)
    img = synth.build_image("phi3mini", seed=1234, spec=spec, context=320)
    _prompt_check(hip, img, synth.prompt(32064, n, seed=7), 320, kv_fp16, [0, 1], split=split)


def test_prefill_attention_512_queries_groups(hip, oracle_threads):  # noqa: F811
    """Four wavefronts a workgroup, query groups of 2, heads of 128."""
    spec = dict(synth.SPECS["small5"], layers=1)
    img = synth.build_image("small5", seed=1234, spec=spec, context=600)
    _prompt_check(hip, img, synth.prompt(32000, 530, seed=7), 600, False, [0])


@pytest.mark.parametrize("t,k", [(Q4_K, 2816), (Q5_K, 256), (Q6_K, 1280), (Q8_0, 1408), (Q8_0, 32), (Q4_0, 4192)])
@pytest.mark.parametrize("m,n,tile", [(2, 129, 32), (32, 300, 32), (33, 96, 64), (64, 2000, 64), (65, 128, 64),
                                      (140, 520, 64), (1030, 140, 128)])
def test_batched_matmul_tiles_and_parts(hip, t, k, m, n, tile):
    """Edges of the 32- and 64-token tiles and a ragged last 128-token tile; K in
    uneven parts, one unit only, and a last unit of fewer than 4 blocks."""
    assert plan(t, m, n, k)[0] == tile
    rng = np.random.default_rng(m + n + k)
    w = random_blocks(t, n, k, m + n)
    a = rng.normal(0, 1, size=(m, k)).astype(np.float32)
    ref = O.matmul(a, w, t, k, n, result_len=m * n).reshape(m, n)
    y = np.zeros(m * n, dtype=np.float32)
    hip.mat_mul(a.reshape(-1), w, y, t, k, n)
    assert row_rel_err(y.reshape(m, n), ref) <= FP32_LEVEL


# heads of 96 at the smallest widths the phi3 mix takes
SMALL96 = dict(synth.SPECS["phi3mini"], hidden=768, layers=2, heads=8, kv_heads=8, ffn=1024, vocab=4096)


@pytest.mark.parametrize("model,t,pos0,kv_fp16,window,splits", [
    ("tiny", 16, 1150, True, 0, 2), ("tiny", 10, 1020, False, 0, 4), ("tiny", 40, 2500, True, 0, 5),
    ("tiny", 5, 8100, True, 0, 16), ("small5", 20, 1080, True, 0, 2), ("small5", 7, 1093, False, 0, 4),
    ("small5", 15, 4000, True, 0, 8), ("small5", 5, 4090, False, 0, 16), ("small96", 2, 1027, True, 0, 2),
    ("small96", 15, 3000, False, 0, 12), ("small96", 33, 4063, True, 0, 8),
    ("tiny", 15, 3000, True, 2100, 4), ("small5", 20, 4070, True, 1500, 3), ("small96", 15, 3000, True, 1100, 2)])
def test_prefill_attention_splits(hip, oracle_threads, model, t, pos0, kv_fp16, window, splits):  # noqa: F811
    """t queries behind pos0 filled keys: the keys over `splits` workgroups as
    well, with ragged last steps, splits without keys for some wavefronts, up to
    three query blocks, and windows whose first key lies far from 0.  Last
    logits and, in the second layer (its rows follow from the first's
    attention), K and V of the new positions."""
    spec = SMALL96 if model == "small96" else dict(synth.SPECS[model], layers=2)
    name = "phi3mini" if model == "small96" else model
    assert host_fn("prefill_attn_splits", "iiiii")(t, pos0, spec["heads"], int(kv_fp16), window) == splits
    ctx = (pos0 + t + 64) // 64 * 64
    img = synth.build_image(name, seed=1234, spec=spec, context=ctx, sliding_window=window)
    prompt = synth.prompt(spec["vocab"], t, seed=7)
    pair = OraclePair(img, kv_fp16, ctx)
    eng = InferenceEngine(LoadedModel.load(img), hip, kv_fp16=kv_fp16, context=ctx)
    try:
        pair.kv_fill_random(pos0, 3)
        eng.kv_fill_random(pos0, 3)
        want = pair.prefill(prompt, pos0)
        got, _ = eng.prefill(prompt, pos0)
        err = float(np.max(np.abs(got - want)))
        worst = floor = 0.0
        for p in range(pos0, pos0 + t):
            rows = list(zip(eng.kv_read(1, p), pair.kv_read(1, p), *pair.kv_alt_reads(1, p)))
            worst = max([worst] + [float(np.max(np.abs(g - r)) / np.max(np.abs(r))) for g, r, *_ in rows])
            floor = max([floor] + [float(np.max(np.abs(o - r)) / np.max(np.abs(r))) for _, r, *alt in rows for o in alt])
        print(f"splits {splits}: max |dlogit| {err:.3e}, KV {worst:.1e} (floor {floor:.1e})")
        assert err <= pair.bounds()[0][0]
        assert worst <= max(KV_MIN, KV_MARGIN * floor)
    finally:
        pair.close()
        eng.dispose()
