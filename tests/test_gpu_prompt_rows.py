"""Prompts through the row-batch pass where they used to run token by token.

Each runtime's prompt pass is compared with the same tokens fed one by one
through the decode step (itself held to the oracle elsewhere), and the states it
leaves behind (K/V, convolution windows, SSM states, position) by the steps that
follow it.
"""
from __future__ import annotations

import numpy as np
import pytest

from chonklm_amd import WORKLOADS, ChonkError, generate_llama_wgsl, load_llama_wgsl_model
from chonklm_amd import runtime
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

LOADERS = {"gpt-webgpu": runtime.load_gpt_wgsl_model, "lfm2-webgpu": runtime.load_lfm_wgsl_model,
           "granite-webgpu": runtime.load_granite_wgsl_model}


def _load(name, synth, **kw):
    md = WORKLOADS[name].model_def(synth(name), **kw)
    return LOADERS.get(md.runtime, load_llama_wgsl_model)(md)


@pytest.mark.parametrize("n", [2, 17, 65])
def test_streamed_prompt_equals_device_loop(n, synth):
    """A streamed call (on_token) and the device loop: the same ids and the same logits."""
    w = WORKLOADS["tiny-qwen3"]
    loaded = _load("tiny-qwen3", synth)
    prompt = np.random.default_rng(n).integers(0, w.spec.vocab, n).tolist()
    want = generate_llama_wgsl(loaded, prompt, 6)["ids"]
    logits = loaded.engine.read_logits()
    runtime.reset_llama_wgsl_conversation(loaded)
    seen = []
    got = generate_llama_wgsl(loaded, prompt, 6, on_token=lambda info: seen.append(info["id"]))["ids"]
    assert got == want == seen
    assert rel_err(loaded.engine.read_logits(), logits) <= 1e-5
    loaded.engine.dispose()


def test_streamed_prompt_past_the_context(synth):
    """A streamed prompt longer than the context fills it, then fails as single steps do."""
    w = WORKLOADS["tiny-qwen3"]
    loaded = _load("tiny-qwen3", synth)
    prompt = np.random.default_rng(3).integers(0, w.spec.vocab, w.max_context + 5).tolist()
    with pytest.raises(ChonkError, match="context exhausted"):
        generate_llama_wgsl(loaded, prompt, 4, on_token=lambda info: None)
    assert loaded.engine.position == w.max_context
    loaded.engine.dispose()
