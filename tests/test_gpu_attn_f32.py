"""k_attn_dec over the fp32 K/V cache against the chunked k_attention it replaces there.

Both read the same cache and accumulate in fp32 in another order; per layer the
attention output differs by at most a few 2^-24 of sums over the positions, so the
logits agree to 2e-5. Positions sit at the edges of the 64-position chunks, inside
and outside Gemma-3's window, and past 128 chunks, where workgroups walk several.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from chonklm_amd import WORKLOADS, _lib, load_llama_wgsl_model
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


def test_fp32_engine_leaves_the_attention_to_an_fp16_engine(synth, monkeypatch):
    """An fp32 engine decodes with k_attn_dec while it is alone, with k_attention beside another
    engine, and with k_attn_dec again afterwards: the logits of the chunked kernel throughout.
    An fp16 engine created beside it has the spin-merging attention all the same."""
    name, ctx = "tiny-qwen3", 400
    monkeypatch.delenv("CHONK_ATTN", raising=False)

    def load(kv):
        md = WORKLOADS[name].model_def(synth(name), kv_dtype=kv)
        md.max_context = ctx
        return load_llama_wgsl_model(md).engine

    def steps(eng, tok):
        out = []
        for _ in range(11):  # (a run of eight steps and more)
            tok = eng.run_token(tok, True)
            out.append(eng.read_logits().copy())
        return out, tok

    def walk(eng, beside):
        eng.fake_context(120, seed=5)
        a, tok = steps(eng, 9)
        with_other = beside()
        b, tok = steps(eng, tok)
        eng.bench_decode(0, 17)  # runs of steps: the multi-step graph
        if with_other:
            with_other.dispose()
        c, tok = steps(eng, tok)
        return a + b + c

    def spin(eng):  # (engine.info is as of the load)
        info = _lib.EngineInfoC()
        _lib.check(_lib.lib().chonk_engine_info_get(eng._h, C.byref(info)), eng._h)
        return info.spin_attention

    eng = load("f32")
    assert spin(eng) == 1
    seen = {}

    def fp16():
        other = load("f16")
        seen.update(fp16=spin(other), fp32=spin(eng))
        other.fake_context(50, seed=1)
        other.run_token(3, True)
        return other

    got = walk(eng, fp16)
    assert seen == dict(fp16=1, fp32=0) and spin(eng) == 1
    eng.dispose()
    monkeypatch.setenv("CHONK_ATTN", "chunked")
    ref = load("f32")
    want = walk(ref, lambda: None)
    ref.dispose()
    for i, (a, b) in enumerate(zip(got, want)):
        assert rel_err(a, b) <= 2e-5, f"step {i}: {rel_err(a, b):.2e}"
