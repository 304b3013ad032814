"""The batched prompt's launches that spread little work over the chip, against
the oracle's sequential loop: RoPE/KV by element groups, attention with the
keys spread over a workgroup's wavefronts, projections in uneven K parts.

Bounds: those of test_gpu_prefill.py (`_prompt_check`).
"""
import numpy as np
import pytest

from dotllm_amd import synth
from test_gpu_prefill import _prompt_check, oracle_threads  # noqa: F401

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
