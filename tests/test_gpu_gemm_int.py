"""The prompt GEMM over integer codes (gemm_int.hip) at the edges of its tiles.

Every weight type through its three tile shapes (128 x 128, 64 x 128 and 64 x 64
weight rows x token rows), with ragged rows (no 16-byte stores), ragged tokens, K
that ends inside a 128-wide stage, and K splits. The bar is relative to float64 in
the 2-norm: the operands carry 22 bits or more and the sums are fp32 over at most
3072 / 32 = 96 matrix steps, sqrt(96) 2^-24 = 6e-7, times up to 8 for the
cancellation between a block's codes and its offset with random scales: 5e-6.
"""
from __future__ import annotations

import numpy as np
import pytest

from chonklm_amd import WORKLOADS, load_llama_wgsl_model
from chonklm_amd.runtime import LlamaWgslBatch
from oracle import oracle as orc
from tests.blocks import TYPES, random_blocks
from tests.conftest import rel_err
from tests.test_gpu_gemm import gpu_gemm
from tests.test_gpu_prompt_rows import _same_state

pytestmark = pytest.mark.gpu

# (weight rows, token rows): 128 x 128 tiles need 256 of them
TILES = [(4100, 1025), (2048, 2047), (257, 513), (515, 600), (130, 65), (1030, 200)]


@pytest.mark.parametrize("n_rows,n_tok", TILES)
@pytest.mark.parametrize("tname,row_len", [("Q4_K", 512), ("Q5_K", 768), ("Q6_K", 512), ("Q8_0", 608), ("Q5_0", 352),
                                           ("Q5_1", 224)])
def test_tiles_of_every_type(tname, row_len, n_rows, n_tok):
    rng = np.random.default_rng(n_rows + n_tok)
    blocks = random_blocks(TYPES[tname], n_rows * row_len, rng)
    w = orc.dequant(TYPES[tname], blocks, n_rows * row_len).reshape(n_rows, row_len).astype(np.float64)
    x = rng.standard_normal((n_tok, row_len)).astype(np.float32)
    got, _ = gpu_gemm(TYPES[tname], blocks, n_rows, row_len, x)
    rows = np.unique(np.r_[0:3, n_tok // 2, n_tok - 17:n_tok])
    want = x[rows].astype(np.float64) @ w.T
    err = np.linalg.norm(got[rows] - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() <= 5e-6, f"{tname}: {err.max():.2e}"


# Bars of the 2-norm against float64, in units of 2^-25 (rms of one rounding; a chain
# of n sums of like size rounds as sqrt(n / 2) of them at the total's size). Codes alone
# (Q8_0, Q5_0): one rounding per 32 k, chains of 8, K / 256 <= 12 of those: sqrt(1 + 4 +
# 6) = 3.3, with the operands' 22 bits 3.6. Q5_1: chains of 12 matrix steps, about four
# roundings each, K / 128 <= 24 of those: sqrt(24 + 12) = 6, with the dropped lo x lo 6.3.
@pytest.mark.parametrize("n_rows,row_len,n_tok", [(1024, 1024, 200), (768, 3072, 200), (576, 576, 48), (3376, 768, 2047),
                                                  (9216, 1024, 300), (130, 160, 515)])
@pytest.mark.parametrize("tname,bar", [("Q8_0", 4.2), ("Q5_0", 4.2), ("Q5_1", 7.0)])
def test_error_of_32_weight_blocks(tname, bar, n_rows, row_len, n_tok):
    rng = np.random.default_rng(n_rows + row_len)
    blocks = random_blocks(TYPES[tname], n_rows * row_len, rng)
    w = orc.dequant(TYPES[tname], blocks, n_rows * row_len).reshape(n_rows, row_len).astype(np.float64)
    x = rng.standard_normal((n_tok, row_len)).astype(np.float32)
    got, _ = gpu_gemm(TYPES[tname], blocks, n_rows, row_len, x)
    rows = np.unique(np.r_[0:16, n_tok // 2, n_tok - 8:n_tok])
    want = x[rows].astype(np.float64) @ w.T
    err = np.linalg.norm(got[rows] - want) / np.linalg.norm(want)
    assert err <= bar * 2.0 ** -25, f"{tname}: {err:.2e}"


# gate | up leave the GEMM as their product where its tiles are 64 x 64 or 128 x 128 and K is
# not split; 64 x 128 tiles leave both
@pytest.mark.parametrize("name,parts", [
    ("qwen3-0.6b-q4_k_m", (300, 600)),   # 64 x 64 (Q4_K, SwiGLU), then 64 x 128; two and four waves per row in the glue
    ("qwen3-0.6b-q4_k_m", (1030,)),      # 128 x 128, six rows in the last tile; a wave per row in the glue
    ("gemma3-270m-q4_k_m", (300,)),      # 64 x 64, Q5_0, GELU
    ("gemma3-270m-q4_k_m", (1301,)),     # 128 x 128, Q5_0, GELU
    ("lfm2.5-350m-q8_0", (601,)),        # 128 x 128, Q8_0
    ("smollm2-135m-q8_0", (1030,)),      # 64 x 128, Q8_0; K ends inside a stage
])
def test_prompt_pass_of_the_workloads_equals_steps(name, parts, synth):
    _same_state(name, parts, synth, max_context=sum(parts) + 8)


def test_step_of_more_than_64_sequences(synth):
    """Over 64 rows a step's GEMMs are the prompt's: the same logits as in a small batch."""
    w = WORKLOADS["tiny-qwen3"]
    eng = load_llama_wgsl_model(w.model_def(synth("tiny-qwen3"))).engine
    rng = np.random.default_rng(8)
    prompts = [rng.integers(0, w.spec.vocab, 3 + s % 5).tolist() for s in range(66)]
    big = LlamaWgslBatch(eng, 66, 16)
    for s, p in enumerate(prompts):
        big.prefill(s, p)
    big.step(list(range(66)), [7] * 66)
    some = [0, 17, 65]
    rows = [big.read_logits(s).copy() for s in some]
    big.close()
    small = LlamaWgslBatch(eng, 3, 16)
    for i, s in enumerate(some):
        small.prefill(i, prompts[s])
    small.step([0, 1, 2], [7] * 3)
    for i in range(3):
        assert rel_err(rows[i], small.read_logits(i)) <= 1e-3  # (fp16 K/V)
    small.close()
    eng.dispose()


@pytest.mark.parametrize("tname", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("n_tok", [1, 16, 17, 32, 33, 64])
def test_head_gemm_token_tiles(tname, n_tok):
    """The lm_head GEMM of a batch with one, two and four token tiles."""
    n_rows, row_len = 32768 + 5, 512
    rng = np.random.default_rng(n_tok)
    blocks = random_blocks(TYPES[tname], n_rows * row_len, rng)
    w = orc.dequant(TYPES[tname], blocks, n_rows * row_len).reshape(n_rows, row_len)
    x = rng.standard_normal((n_tok, row_len)).astype(np.float32)
    got, _ = gpu_gemm(TYPES[tname], blocks, n_rows, row_len, x)
    rows = np.unique([0, n_tok // 2, n_tok - 1])
    want = x[rows].astype(np.float64) @ w.T.astype(np.float64)
    err = np.linalg.norm(got[rows] - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() <= 5e-6, f"{tname}: {err.max():.2e}"


def test_step_rows_do_not_depend_on_the_batch(synth):
    """1 to 40 rows (one, two and four token tiles): a row's logits are the same."""
    w = WORKLOADS["tiny-qwen3"]
    eng = load_llama_wgsl_model(w.model_def(synth("tiny-qwen3"))).engine
    rng = np.random.default_rng(9)
    prompts = [rng.integers(0, w.spec.vocab, 3 + s % 5).tolist() for s in range(40)]
    batch = LlamaWgslBatch(eng, 40, 16)
    want = None
    for n in (40, 33, 32, 17, 16, 2, 1):
        for s in range(n):
            batch.prefill(s, prompts[s])
        batch.step(list(range(n)), [7] * n)
        rows = np.stack([batch.read_logits(s) for s in range(n)])
        assert np.isfinite(rows).all()
        want = rows if want is None else want
        # (fp32 sums in another order at most: the attention splits few rows' pages)
        assert rel_err(rows, want[:n]) <= 2e-5, f"{n} rows"
    batch.close()
    eng.dispose()
