"""k_attn_dec over the fp32 K/V cache against the chunked k_attention it replaces there.

Both read the same cache and accumulate in fp32 in another order; per layer the
attention output differs by at most a few 2^-24 of sums over the positions, so the
logits agree to 2e-5. Positions sit at the edges of the 64-position chunks, inside
and outside Gemma-3's window, and past 128 chunks, where workgroups walk several.
"""
from __future__ import annotations

import numpy as np
import pytest

from chonklm_amd import WORKLOADS, load_llama_wgsl_model
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu


def _steps(synth, name, ctx, positions):
    md = WORKLOADS[name].model_def(synth(name), kv_dtype="f32")
    md.max_context = ctx
    eng = load_llama_wgsl_model(md).engine
    out = []
    for pos in positions:
        eng.fake_context(pos, seed=pos + 1)
        for tok in (17, 23):  # the second step reads the row the first one wrote
            eng.run_token(tok, True)
            out.append(eng.read_logits().copy())
    info = eng.info
    eng.dispose()
    return info, out


@pytest.mark.parametrize("name,ctx,positions", [
    ("tiny-qwen3", 400, (0, 1, 62, 63, 64, 65, 127, 300)),        # head_dim 64, pairs of heads
    ("tiny-qwen3-hd128", 400, (0, 63, 64, 200, 397)),
    ("tiny-gemma3", 160, (0, 5, 63, 64, 100)),                    # head_dim 256, sliding window
    ("smollm2-135m-q8_0", 512, (33, 500)),                        # groups of three
    ("qwen3-0.6b-q4_k_m", 9000, (4000, 8300)),                    # two sub-chunks per workgroup
])
def test_fp32_decode_attention_equals_chunked(name, ctx, positions, synth, monkeypatch):
    monkeypatch.delenv("CHONK_ATTN", raising=False)
    info, got = _steps(synth, name, ctx, positions)
    monkeypatch.setenv("CHONK_ATTN", "chunked")
    ref_info, want = _steps(synth, name, ctx, positions)
    assert info["spin_attention"] == 1 and ref_info["spin_attention"] == 0
    for i, (a, b) in enumerate(zip(got, want)):
        assert np.isfinite(a).all()
        assert rel_err(a, b) <= 2e-5, f"step {i}: {rel_err(a, b):.2e}"
