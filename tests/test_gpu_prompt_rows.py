"""Prompts through the row-batch pass, and streamed prompts token by token.

Each runtime's prompt pass is compared with the same tokens fed one by one
through the decode step (itself held to the oracle elsewhere), and the states it
leaves behind (K/V, convolution windows, SSM states, position) by the steps that
follow it.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from chonklm_amd import WORKLOADS, ChonkError, generate_llama_wgsl, load_llama_wgsl_model
from chonklm_amd import runtime, write_synthetic_gguf
from chonklm_amd.registry import SynthSpec, Workload
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

LOADERS = {"gpt-webgpu": runtime.load_gpt_wgsl_model, "lfm2-webgpu": runtime.load_lfm_wgsl_model,
           "granite-webgpu": runtime.load_granite_wgsl_model}


def _load(name, synth, **kw):
    md = WORKLOADS[name].model_def(synth(name), **kw)
    return LOADERS.get(md.runtime, load_llama_wgsl_model)(md)


GENERATE = {"gpt-webgpu": runtime.generate_gpt_wgsl, "lfm2-webgpu": runtime.generate_lfm_wgsl,
            "granite-webgpu": runtime.generate_granite_wgsl}


@pytest.mark.parametrize("name,n,new", [("tiny-qwen3", 2, 6), ("tiny-qwen3", 65, 6), ("tiny-gpt2", 65, 6),
                                        ("tiny-lfm2", 65, 6), ("tiny-granite", 65, 6), ("qwen3-0.6b-q4_k_m", 301, 16)])
def test_streamed_call_equals_single_steps(name, n, new, synth):
    """A streamed call (on_token) is run_token by run_token: the same ids, the logits to the bit.

    (Through row batches some fp16 K/V values round the other way, which moves the
    logits by 1e-4 and now and then the greedy id at a near tie.)"""
    w = WORKLOADS[name]
    loaded = _load(name, synth)
    eng = loaded.engine
    prompt = np.random.default_rng(n).integers(0, w.spec.vocab, n).tolist()
    for t in prompt[:-1]:
        eng.run_token(t, False)
    want = [eng.run_token(prompt[-1], True)]
    while len(want) < new and want[-1] not in w.eos_ids:
        want.append(eng.run_token(want[-1], True))
    if loaded.runtime in GENERATE and want[-1] not in w.eos_ids:
        eng.run_token(want[-1], True)  # (these loops also run the last id)
    logits = eng.read_logits().copy()
    eng.reset()
    seen = []
    generate = GENERATE.get(loaded.runtime, generate_llama_wgsl)
    got = generate(loaded, prompt, new, on_token=lambda info: seen.append(info["id"]))["ids"]
    assert got == want == seen
    assert (eng.read_logits() == logits).all()
    eng.dispose()


def test_streamed_prompt_past_the_context(synth):
    """A streamed prompt longer than the context fills it, then fails as single steps do."""
    w = WORKLOADS["tiny-qwen3"]
    loaded = _load("tiny-qwen3", synth)
    prompt = np.random.default_rng(3).integers(0, w.spec.vocab, w.max_context + 5).tolist()
    with pytest.raises(ChonkError, match="context exhausted"):
        generate_llama_wgsl(loaded, prompt, 4, on_token=lambda info: None)
    assert loaded.engine.position == w.max_context
    loaded.engine.dispose()


def _same_state(name, parts, synth, max_context=None):
    """prefill of each part in turn, against the same tokens one by one: the logits of
    the next two steps. With the fp32 cache both sides are fp32-class sums of the same
    values in another order: 3e-7 apart per layer at most, over at most 32 layers and
    two linear branches each, so 2e-5 bounds them."""
    w = name if isinstance(name, Workload) else WORKLOADS[name]
    md = w.model_def(synth(name), kv_dtype="f32")
    if max_context:
        md.max_context = max_context
    tokens = np.random.default_rng(sum(parts)).integers(0, w.spec.vocab, sum(parts) + 2).tolist()
    loaded = LOADERS.get(md.runtime, load_llama_wgsl_model)(md)
    eng = loaded.engine
    out = []
    for rows in (True, False):
        eng.reset()
        at = 0
        for n in parts:
            if rows:
                eng.prefill(tokens[at:at + n])
            else:
                for t in tokens[at:at + n]:
                    eng.run_token(t, False)
            at += n
        assert eng.position == at
        got = []
        for t in tokens[at:]:
            eng.run_token(t, True)
            got.append(eng.read_logits().copy())
        out.append(got)
    eng.dispose()
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert rel_err(a, b) <= 2e-5


# windows of two (lfm2) and three (granite) earlier inputs, the scan's 32 staged
# rows, 64-row GEMM tiles; an odd and an even first part (the Mamba2 window's parity)
@pytest.mark.parametrize("parts", [(1,), (2,), (3,), (1, 1, 2), (3, 32), (4, 33), (64, 1), (65, 64)])
@pytest.mark.parametrize("name", ["tiny-gpt2", "tiny-lfm2", "tiny-lfm2-q8", "tiny-granite", "tiny-granite-q8"])
def test_prompt_rows_equal_steps(name, parts, synth):
    _same_state(name, parts, synth)


@pytest.mark.parametrize("name", ["tiny-lfm2", "tiny-granite"])
def test_prompt_of_two_passes_equals_steps(name, synth):
    """2051 + 6 rows: the states cross the 2048-row pass boundary and a call's."""
    _same_state(name, (2051, 6), synth, max_context=2200)


@pytest.mark.parametrize("name", ["lfm2.5-350m-q4_k_m", "openelm-270m-q4_k_m", "granite-4.0-h-350m-q8_0"])
def test_prompt_rows_of_the_workload_shapes_equal_steps(name, synth):
    """Feed-forward rows over 4096 elements (eight per thread) and 48 SSM heads."""
    _same_state(name, (70, 3), synth)


@pytest.mark.parametrize("recipe", ["q4_k_m", "q8_0"])
@pytest.mark.parametrize("heads,kv_heads", [(6, 3), (4, 1), (6, 2), (3, 1)])
def test_prompt_rows_of_32_wide_heads_equal_steps(heads, kv_heads, recipe, tmp_path):
    """q and k in one GEMM where k (32 or 96 rows) ends inside a 64-row tile; one row tile and several."""
    spec = SynthSpec(arch="llama", recipe=recipe, hidden=256, layers=3, heads=heads, kv_heads=kv_heads, head_dim=32,
                     ffn=512, vocab=600, context_length=512, seed=heads)
    w = Workload("heads32", spec, max_context=300, eos_ids=[2], prompt_tokens=8, decode_tokens=8)
    path = write_synthetic_gguf(w, str(tmp_path / "m.gguf"))
    _same_state(w, (17, 200), lambda _: path)


@pytest.mark.parametrize("name", ["tiny-gpt2", "tiny-lfm2", "tiny-granite", "openelm-270m-q4_k_m"])
def test_one_or_two_tokens_are_steps(name, synth):
    """Prompts of one and two tokens run as decode steps on these runtimes: the logits to the bit."""
    w = WORKLOADS[name]
    eng = _load(name, synth).engine
    tokens = np.random.default_rng(1).integers(0, w.spec.vocab, 20).tolist()
    for n in (1, 2):
        got = []
        for rows in (True, False):
            eng.reset()
            for t in tokens[:9]:
                eng.run_token(t, False)
            if rows:
                eng.prefill(tokens[9:9 + n])
            else:
                for t in tokens[9:9 + n]:
                    eng.run_token(t, False)
            assert eng.position == 9 + n
            eng.run_token(tokens[15], True)
            got.append(eng.read_logits().copy())
        assert (got[0] == got[1]).all(), f"{n} tokens"
    eng.dispose()


@pytest.mark.parametrize("more", [1, 2, 3])
@pytest.mark.parametrize("name", ["tiny-gpt2", "tiny-lfm2", "tiny-granite"])
def test_continued_conversation_equals_steps(name, more, synth):
    """A second call whose prompt adds one to three tokens to the first call's: the ids and
    logits of run_token over those tokens, to the bit."""
    w = WORKLOADS[name]
    loaded = _load(name, synth)
    eng, generate = loaded.engine, GENERATE[loaded.runtime]
    rng = np.random.default_rng(more)
    first = rng.integers(0, w.spec.vocab, 12).tolist()
    talk = first + generate(loaded, first, 4)["ids"]
    added = rng.integers(0, w.spec.vocab, more).tolist()
    got = generate(loaded, talk + added, 3)["ids"]
    logits = eng.read_logits().copy()
    eng.reset()
    eng.prefill(first[:-1])
    for t in first[-1:] + talk[len(first):] + added[:-1]:
        eng.run_token(t, False)
    want = [eng.run_token(added[-1], True)]
    while len(want) < 3 and want[-1] not in w.eos_ids:
        want.append(eng.run_token(want[-1], True))
    if want[-1] not in w.eos_ids:
        eng.run_token(want[-1], True)  # (these loops also run the last id)
    assert got == want
    assert (eng.read_logits() == logits).all()
    eng.dispose()


def _free_mib():
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value / 2 ** 20


# MiB of a short prompt's buffers: 256 rows of (x, q|k|v, attention, block sums, two planes)
# floats or halves, and the partial sums of 2048 rows of the widest result, 2 ffn (or in_proj)
@pytest.mark.parametrize("name,most", [("gpt2-124m-q4_k_m", 60), ("lfm2.5-350m-q4_k_m", 90),
                                       ("openelm-270m-q4_k_m", 100), ("qwen3-0.6b-q4_k_m", 70)])
def test_short_prompts_take_little_memory(name, most, synth):
    w = WORKLOADS[name]
    eng = _load(name, synth).engine
    tokens = np.random.default_rng(1).integers(0, w.spec.vocab, 20).tolist()
    eng.run_token(tokens[0], True)
    before = _free_mib()
    eng.prefill(tokens)
    assert before - _free_mib() <= most
    eng.dispose()


@pytest.mark.parametrize("name", ["tiny-qwen3", "tiny-lfm2", "tiny-granite-q8"])
def test_longer_prompts_make_the_buffers_larger(name, synth):
    """20, 300 and 900 rows: each call's buffers replace smaller ones; the states stay."""
    _same_state(name, (20, 300, 900), synth, max_context=1300)
