"""The batched prompt's launches that spread little work over the chip, against
the oracle's sequential loop: RoPE/KV by element groups, attention with the
keys spread over a workgroup's wavefronts, projections in uneven K parts.

Bounds: those of test_gpu_prefill.py (`_prompt_check`).
"""
import numpy as np
import pytest

from dotllm_amd import Q4_0, Q4_K, Q5_K, Q6_K, Q8_0, synth
from oracle import oracle as O
from test_gpu_prefill import FP32_LEVEL, _prompt_check, oracle_threads, random_blocks, row_rel_err  # noqa: F401

pytestmark = pytest.mark.gpu


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
@pytest.mark.parametrize("m,n", [(2, 129), (32, 300), (33, 96), (64, 2000), (65, 128), (140, 520)])
def test_batched_matmul_tiles_and_parts(hip, t, k, m, n):
    """Edges of the 32-, 64- and 128-token tiles; K in uneven parts, one unit
    only, and a last unit of fewer than 4 blocks."""
    rng = np.random.default_rng(m + n + k)
    w = random_blocks(t, n, k, m + n)
    a = rng.normal(0, 1, size=(m, k)).astype(np.float32)
    ref = O.matmul(a, w, t, k, n, result_len=m * n).reshape(m, n)
    y = np.zeros(m * n, dtype=np.float32)
    hip.mat_mul(a.reshape(-1), w, y, t, k, n)
    assert row_rel_err(y.reshape(m, n), ref) <= FP32_LEVEL


@pytest.mark.parametrize("model,n,split,kv_fp16", [("tiny", 1030, 1029, True), ("tiny", 1030, 1020, False),
                                                   ("phi3mini", 560, 545, True), ("small5", 1100, 1093, False),
                                                   ("small5", 1100, 1080, True)])
def test_prefill_attention_splits(hip, oracle_threads, model, n, split, kv_fp16):  # noqa: F811
    """A few queries behind many keys: the keys over 2 to 8 workgroups as well,
    some splits without keys for a wavefront."""
    spec = dict(synth.SPECS[model], layers=1)
    img = synth.build_image(model, seed=1234, spec=spec, context=1120)
    _prompt_check(hip, img, synth.prompt(32000, n, seed=7), 1120, kv_fp16, [0], split=split)


def test_prefill_attention_splits_window(hip):
    """The same with a window: splits start at its first key."""
    img = synth.build_image("tiny", seed=1234, context=1120, sliding_window=700)
    _prompt_check(hip, img, synth.prompt(32000, 1000, seed=7), 1120, True, [0, 3], split=985)
