"""The work that a program using this framework gives it, as measurable cases.

A program loads one model (a GGUF file) and then calls one of three things, over
and over, with prompts of all lengths:

  generate   a chat turn: prompt in, new token ids out (generate_*_wgsl), either
             as one device-driven call or streamed token by token
  guided     the host drives the loop itself (reset, prefill, run_token): a
             grammar or a known continuation fixes each token, the logits are read
  batch      many independent sequences served together (LlamaWgslBatch)

The models are the workloads of the package's registry (random weights of those
shapes). A model's weights are the same whatever the seed, as a user's are; the
seed makes the prompts, the forced tokens and the sampler's seed. One model is
loaded at a time, as in a program that serves one, and stays loaded for as long
as the cases ask for it.

``exact`` evaluates the same decoders in float64 with plain torch from the GGUF
file's bytes (K/V rounded to the cache's type, which the program chose).
"""
from __future__ import annotations

import os
import struct
import tempfile
from typing import Optional

import numpy as np
import torch

from chonklm_amd import runtime as rt_api
from chonklm_amd.registry import WORKLOADS

LLAMA_FAMILY = ("smollm2-135m-q4_k_m", "smollm2-135m-q8_0", "qwen3-0.6b-q4_k_m", "gemma3-270m-q4_k_m")
SAMPLING = dict(temperature=0.8, top_k=40)  # the sampled workload's options


# ---- the cases ------------------------------------------------------------------

def _case(kind, model, prompt, new, context, kv="f16", stream=False, sample=False, seqs=1, name=None):
    c = dict(kind=kind, model=model, prompt=prompt, new=new, context=context, kv=kv, stream=stream, sample=sample,
             seqs=seqs)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: first token of a short question (launches and latency)
        _case("guided", "smollm2-135m-q4_k_m", 7, 1, 512, name="first_token_smollm2"),
        # grammar-guided decoding of a small model, 8-bit weights, fp32 K/V
        _case("guided", "smollm2-135m-q8_0", 33, 24, 512, kv="f32", name="guided_smollm2_q8_f32kv"),
        # a streamed chat turn (on_token), the reference's own way of calling
        _case("generate", "qwen3-0.6b-q4_k_m", 301, 16, 2304, stream=True, name="stream_qwen3"),
        # time to first token of a long question
        _case("guided", "qwen3-0.6b-q4_k_m", 2048, 1, 2304, name="prompt_qwen3_2k"),
        # a whole chat turn on the device: long prompt, then decoding at 2K context
        _case("generate", "qwen3-0.6b-q4_k_m", 2048, 32, 2304, name="generate_qwen3_2k"),
        # a document of odd length, then decoding at long context (the largest)
        _case("guided", "qwen3-0.6b-q4_k_m", 11003, 16, 16384, name="document_qwen3_11k"),
        # sampled chat turn; sliding windows, 256-wide heads, 262144 ids
        _case("generate", "gemma3-270m-q4_k_m", 1024, 24, 1152, sample=True, name="sample_gemma3_1k"),
        # serving: a batch of ragged requests admitted, then decoded together
        _case("batch", "qwen3-0.6b-q4_k_m", 512, 24, 2304, seqs=64, name="batch_qwen3_64"),
        # serving a few short requests with a small model
        _case("batch", "smollm2-135m-q8_0", 61, 40, 512, seqs=5, name="batch_smollm2_5"),
        # chat turns on the other runtimes: short convolutions, Mamba2, GPT-2
        _case("generate", "lfm2.5-350m-q4_k_m", 201, 24, 4096, name="chat_lfm2"),
        _case("generate", "granite-4.0-h-350m-q8_0", 150, 16, 4096, name="chat_granite_q8"),
        _case("generate", "gpt2-124m-q4_k_m", 512, 24, 1024, name="chat_gpt2"),
    ]


def draw(rng):
    """One more case of the same ranges."""
    def log_int(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["generate", "generate", "guided", "batch"])
    if kind == "batch":
        model = rng.choice(LLAMA_FAMILY)
        seqs, prompt, new = log_int(2, 64), log_int(8, 512), log_int(4, 24)
        return _case("batch", model, prompt, new, 2304 if "qwen3" in model else 1152, seqs=seqs)
    model = rng.choice(LLAMA_FAMILY + ("qwen3-0.6b-q4_k_m", "openelm-270m-q4_k_m", "gpt2-124m-q4_k_m",
                                       "lfm2.5-350m-q4_k_m", "lfm2.5-350m-q8_0", "granite-4.0-h-350m-q4_k_m",
                                       "granite-4.0-h-350m-q8_0"))
    most = {"qwen3-0.6b-q4_k_m": 8192, "gpt2-124m-q4_k_m": 900, "lfm2.5-350m-q4_k_m": 600, "lfm2.5-350m-q8_0": 600,
            "granite-4.0-h-350m-q4_k_m": 400, "granite-4.0-h-350m-q8_0": 400}.get(model, 1900)
    stream = kind == "generate" and rng.random() < 0.35
    kv = "f32" if rng.random() < 0.15 else "f16"
    prompt = log_int(3, min(most, 500) if stream else min(most, 1900) if kv == "f32" else most)
    new = log_int(1, 24)
    context = {"gpt2-124m-q4_k_m": 1024, "openelm-270m-q4_k_m": 2048}.get(
        model, 512 if prompt < 480 else 2304 if prompt < 2200 else 16384)
    if "granite" in model or "lfm2" in model:
        context = 4096
    sample = kind == "generate" and model in LLAMA_FAMILY and rng.random() < 0.25
    return _case(kind, model, prompt, new, context, kv=kv, stream=stream, sample=sample)


# ---- the calls ------------------------------------------------------------------

class _Live:
    """The model a serving program has loaded, and its batch of sequences."""

    key: Optional[tuple] = None
    loaded = None
    batch_key: Optional[tuple] = None
    batch = None


_live = _Live()


def _model_file(model: str) -> str:
    d = os.path.join(tempfile.gettempdir(), f"chonk_models_{os.getuid()}")
    os.makedirs(d, exist_ok=True)
    path = os.path.join(d, f"{model}.gguf")
    if not os.path.exists(path):
        part = f"{path}.{os.getpid()}"
        rt_api.write_synthetic_gguf(model, part)
        os.replace(part, path)
    return path


def _load(case):
    key = (case["model"], case["context"], case["kv"])
    if _live.key != key:
        if _live.batch is not None:
            _live.batch.close()
        if _live.loaded is not None:
            _live.loaded.engine.dispose()
        _live.batch = _live.batch_key = _live.loaded = None
        md = WORKLOADS[case["model"]].model_def(_model_file(case["model"]), kv_dtype=case["kv"])
        md.max_context = case["context"]
        load = {"gpt-webgpu": rt_api.load_gpt_wgsl_model, "lfm2-webgpu": rt_api.load_lfm_wgsl_model,
                "granite-webgpu": rt_api.load_granite_wgsl_model}.get(md.runtime, rt_api.load_llama_wgsl_model)
        _live.loaded, _live.key = load(md), key
    return _live.loaded


def _tokens(case, seed):
    """The prompts (one per sequence, ragged in a batch) and the forced tokens [new][seqs]."""
    rng = np.random.default_rng([int(seed), case["prompt"], case["seqs"]])
    vocab = WORKLOADS[case["model"]].spec.vocab
    n = [case["prompt"]] * case["seqs"]
    if case["kind"] == "batch":
        n = [int(x) for x in rng.integers(max(1, case["prompt"] // 8), case["prompt"] + 1, case["seqs"])]
        n[0] = case["prompt"]
    prompts = [rng.integers(0, vocab, k).tolist() for k in n]
    forced = rng.integers(0, vocab, (case["new"], case["seqs"])).tolist()
    return prompts, forced


def prepare(case, seed):
    prompts, forced = _tokens(case, seed)
    loaded = _load(case)
    state = dict(case=case, seed=int(seed), loaded=loaded, prompts=prompts, forced=forced)
    if case["kind"] == "batch":
        key = (case["seqs"], case["prompt"] + case["new"])
        if _live.batch_key != key:
            if _live.batch is not None:
                _live.batch.close()
            _live.batch = rt_api.LlamaWgslBatch(loaded.engine, *key)
            _live.batch_key = key
        state["batch"] = _live.batch
    return state


def run(state):
    case, loaded = state["case"], state["loaded"]
    engine = loaded.engine
    if case["kind"] == "generate":
        kw = dict(SAMPLING, seed=state["seed"]) if case["sample"] else {}
        if case["stream"]:
            streamed = []
            kw["on_token"] = streamed.append
        generate = {"gpt-webgpu": rt_api.generate_gpt_wgsl, "lfm2-webgpu": rt_api.generate_lfm_wgsl,
                    "granite-webgpu": rt_api.generate_granite_wgsl}.get(loaded.runtime, rt_api.generate_llama_wgsl)
        rt_api.reset_llama_wgsl_conversation(loaded)
        out = generate(loaded, state["prompts"][0], case["new"], **kw)
        return {"ids": np.asarray(out["ids"], dtype=np.int64), "logits": engine.read_logits()}
    if case["kind"] == "guided":
        prompt = state["prompts"][0]
        engine.reset()
        if len(prompt) > 1:
            engine.prefill(prompt[:-1])
        engine.run_token(prompt[-1], True)
        for step in state["forced"][: case["new"] - 1]:
            engine.run_token(step[0], True)
        return {"logits": engine.read_logits()}
    batch, seqs = state["batch"], list(range(case["seqs"]))
    for s, prompt in enumerate(state["prompts"]):
        batch.prefill(s, prompt)
    for step in state["forced"]:
        batch.step(seqs, step)
    return {"logits": np.stack([batch.read_logits(s) for s in seqs])}


def tolerance(case):
    # Measured against float64 over these ranges: 4e-7 with fp32 K/V; with fp16
    # K/V up to 2.4e-4 (the 256-wide heads; 2e-5 .. 1e-4 elsewhere), because a
    # K/V value that rounds the other way moves the logits by far more than
    # fp32 sums in another order do.
    return {"rel": 1e-5 if case["kv"] == "f32" else 1e-3}


# ---- what a pass cannot do without ---------------------------------------------------

def work(case):
    spec = WORKLOADS[case["model"]].spec
    prompts, _ = _tokens(case, 0)
    H, hd = spec.hidden, spec.head_dim or spec.hidden // spec.heads
    per_weight = 1.0625 if spec.recipe == "q8_0" else 0.6
    heads = spec.layer_heads or [spec.heads] * spec.layers
    kvh = spec.layer_kv_heads or [spec.kv_heads] * spec.layers
    ffn = spec.layer_ffn or [spec.ffn] * spec.layers
    linear, kv_row, attn = 0, 0, []  # weights; K/V bytes per position; per attention layer (q width, window)
    for i in range(spec.layers):
        linear += (2 if spec.arch == "gpt2" else 3) * H * ffn[i]
        if kvh[i] == 0 and spec.arch == "lfm2":
            linear += 4 * H * H
        elif kvh[i] == 0:
            linear += H * (4 * H + 256 + 2 * H // 32) + 2 * H * H  # Mamba2 blocks: inner size 2 H
        else:
            linear += H * hd * (2 * heads[i] + 2 * kvh[i])
            kv_row += 2 * kvh[i] * hd * (4 if case["kv"] == "f32" else 2)
            attn.append((heads[i] * hd, spec.sliding_window if spec.sliding_window and i % 6 != 5 else 0))
    head = spec.vocab * H
    w_bytes, h_bytes = linear * per_weight, head * (1.0625 if spec.recipe == "q8_0" else 0.82)
    steps = case["new"] if case["kind"] == "batch" else max(0, case["new"] - 1)
    flops = bytes_ = 0.0
    for p in prompts:
        n = len(p) + steps
        flops += 2.0 * linear * n + 2.0 * head * (steps + 1)
        for width, window in attn:
            seen = sum(min(t + 1, window or t + 1) for t in range(n))
            flops += 4.0 * width * seen
        bytes_ += kv_row * n + sum(kv_row * (len(p) + s) for s in range(steps)) + kv_row * len(p)
    passes = len(prompts) if case["kind"] == "batch" else 1  # prompts arrive one by one
    bytes_ += passes * (w_bytes + h_bytes) + steps * (w_bytes + h_bytes) + 4.0 * spec.vocab * case["seqs"]
    return {"bytes": bytes_, "flops": flops}


# ---- float64 ------------------------------------------------------------------------

F64 = torch.float64


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _half(b):  # uint8 [n, 2] -> float64 [n, 1]
    return b.contiguous().view(torch.float16).to(F64)


def _decode_blocks(kind, raw):
    """GGUF block bytes (uint8, 1-D) -> float64 values (Q8_0, Q5_0, Q4_K, Q5_K, Q6_K, F32, F16)."""
    if kind == 0:
        return raw.view(torch.float32).to(F64)
    if kind == 1:
        return raw.view(torch.float16).to(F64)
    if kind == 8:
        b = raw.view(-1, 34)
        return (b[:, 2:].contiguous().view(torch.int8).to(F64) * _half(b[:, :2])).reshape(-1)
    if kind == 6:
        b = raw.view(-1, 22).to(torch.int32)
        bits = (b[:, 2:6, None] >> torch.arange(8, device=raw.device)) & 1
        q = torch.cat([b[:, 6:] & 15, b[:, 6:] >> 4], 1) + 16 * bits.reshape(-1, 32) - 16
        return (q.to(F64) * _half(raw.view(-1, 22)[:, :2])).reshape(-1)
    if kind in (12, 13):
        b = raw.view(-1, 144 if kind == 12 else 176)
        s = b[:, 4:16].to(torch.int32)
        low, high, tail = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat([low & 63, (tail & 15) | ((low >> 6) << 4)], 1).to(F64)
        mn = torch.cat([high & 63, (tail >> 4) | ((high >> 6) << 4)], 1).to(F64)
        q = b[:, -128:].reshape(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32)
        if kind == 13:
            bit = torch.arange(8, device=raw.device, dtype=torch.uint8).view(1, 8, 1)
            q = q | (((b[:, 16:48].reshape(-1, 1, 32) >> bit) & 1) << 4)
        q = q.to(F64)
        return (q * (_half(b[:, :2]) * sc)[:, :, None] - (_half(b[:, 2:4]) * mn)[:, :, None]).reshape(-1)
    if kind == 14:
        b = raw.view(-1, 210)
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32).to(torch.int32), b[:, 128:192].reshape(-1, 2, 1, 32).to(torch.int32)
        q = torch.cat([ql & 15, ql >> 4], 2) | (((qh >> torch.tensor([0, 2, 4, 6], device=raw.device).view(1, 1, 4, 1))
                                                & 3) << 4)
        sc = b[:, 192:208].contiguous().view(torch.int8).to(F64).view(-1, 16, 1)
        return ((q - 32).reshape(-1, 16, 16).to(F64) * sc * _half(b[:, 208:])[:, :, None]).reshape(-1)
    raise ValueError(f"GGUF tensor type {kind}")


_BLOCK = {0: (1, 4), 1: (1, 2), 6: (32, 22), 8: (32, 34), 12: (256, 144), 13: (256, 176), 14: (256, 210)}


def _read_gguf(path):
    """{name: float64 tensor on the device}; matrices are [rows][row length]."""
    raw = np.memmap(path, dtype=np.uint8, mode="r")
    at = 0

    def take(fmt):
        nonlocal at
        v = struct.unpack_from("<" + fmt, raw, at)[0]
        at += struct.calcsize("<" + fmt)
        return v

    def text():
        nonlocal at
        n = take("Q")
        at += n
        return bytes(raw[at - n:at]).decode()

    def value(kind):
        if kind == 8:
            return text()
        if kind == 9:
            item = take("I")
            return [value(item) for _ in range(take("Q"))]
        return take({0: "B", 1: "b", 2: "H", 3: "h", 4: "I", 5: "i", 6: "f", 7: "?", 10: "Q", 11: "q", 12: "d"}[kind])

    if take("I") != 0x46554747:
        raise ValueError("not a GGUF file")
    take("I")
    n_tensors, n_keys = take("Q"), take("Q")
    for _ in range(n_keys):
        text()
        value(take("I"))
    table = []
    for _ in range(n_tensors):
        name = text()
        shape = [take("Q") for _ in range(take("I"))]
        table.append((name, shape, take("I"), take("Q")))
    base = (at + 31) // 32 * 32
    out = {}
    for name, shape, kind, offset in table:
        elems, size = _BLOCK[kind]
        n = int(np.prod(shape)) // elems * size
        data = torch.from_numpy(np.array(raw[base + offset:base + offset + n])).to(_device())
        out[name] = _decode_blocks(kind, data).view(*reversed(shape))
    return out


class _Exact:
    """The registry's decoders over rows of tokens, in float64."""

    CHUNK = 1024  # rows per pass (bounds the attention scores)

    def __init__(self, model, kv):
        self.spec, self.kv = WORKLOADS[model].spec, kv
        self.w = _read_gguf(_model_file(model))
        self.arch = self.spec.arch
        self.eps = 1e-5 if self.arch in ("lfm2", "granitehybrid") else self.spec.norm_eps
        self.hd = self.spec.head_dim or self.spec.hidden // self.spec.heads
        self.reset()

    def reset(self):
        L = self.spec.layers
        self.pos = 0
        self.k, self.v = [[] for _ in range(L)], [[] for _ in range(L)]
        self.past = [None] * L   # convolution inputs of the last positions
        self.state = [None] * L  # Mamba2 states

    # -- pieces
    def _norm(self, x, name, eps=None):
        if self.arch == "gpt2":
            x = x - x.mean(-1, keepdim=True)
        y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + (self.eps if eps is None else eps)) * self.w[name + ".weight"]
        return y + self.w[name + ".bias"] if self.arch == "gpt2" else y

    def _linear(self, x, name):
        y = x @ self.w[name + ".weight"].T
        return y + self.w[name + ".bias"] if self.arch == "gpt2" else y

    def _rope(self, x, theta):
        half = self.hd // 2
        inv = theta ** (-2.0 * torch.arange(half, device=x.device, dtype=F64) / self.hd)
        ang = (self.pos + torch.arange(x.shape[0], device=x.device, dtype=F64))[:, None, None] * inv
        co, si = torch.cos(ang), torch.sin(ang)
        if self.arch == "llama":
            a, b = x[..., 0::2], x[..., 1::2]
            return torch.stack([a * co - b * si, a * si + b * co], -1).reshape(x.shape)
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * co - b * si, a * si + b * co], -1)

    def _gelu(self, x):
        g = 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))
        return torch.where(x > 10, x, torch.where(x < -10, torch.zeros_like(x), g))

    def _attention(self, i, n):
        b, hd, T = f"blk.{i}.", self.hd, n.shape[0]
        spec = self.spec
        nh = spec.layer_heads[i] if spec.layer_heads else spec.heads
        nkv = spec.layer_kv_heads[i] if spec.layer_kv_heads else spec.kv_heads
        if b + "attn_qkv.weight" in self.w:
            q, k, v = self._linear(n, b + "attn_qkv").split([nh * hd, nkv * hd, nkv * hd], -1)
        else:
            q, k, v = (self._linear(n, b + "attn_" + c) for c in "qkv")
        q, k, v = q.reshape(T, nh, hd), k.reshape(T, nkv, hd), v.reshape(T, nkv, hd)
        if b + "attn_q_norm.weight" in self.w:
            q, k = self._norm(q, b + "attn_q_norm"), self._norm(k, b + "attn_k_norm")
        window = 0
        theta = {"lfm2": 1e6, "granitehybrid": 0, "gpt2": 0}.get(self.arch, spec.rope_theta)
        if self.arch == "gemma3" and i % 6 != 5:
            theta, window = 10000.0, spec.sliding_window
        if theta:
            q, k = self._rope(q, theta), self._rope(k, theta)
        if self.kv == "f16":
            k, v = k.to(torch.float16).to(F64), v.to(torch.float16).to(F64)
        self.k[i].append(k)
        self.v[i].append(v)
        k, v = torch.cat(self.k[i]), torch.cat(self.v[i])
        scale = 1.0 / 64 if self.arch == "granitehybrid" else hd ** -0.5
        row = self.pos + torch.arange(T, device=n.device)[:, None]
        col = torch.arange(k.shape[0], device=n.device)[None]
        hide = (col > row) | ((col <= row - window) if window else torch.zeros_like(col > row))
        out = torch.empty_like(q)
        for h in range(nh):
            g = h // (nh // nkv)
            s = (q[:, h] @ k[:, g].T.contiguous()) * scale
            out[:, h] = torch.softmax(s.masked_fill(hide, float("-inf")), -1) @ v[:, g].contiguous()
        return self._linear(out.reshape(T, nh * hd), b + "attn_output")

    def _taps(self, i, x, taps):
        """Causal convolution of the rows x with taps [channels][n], over the earlier rows."""
        n = taps.shape[1]
        past = self.past[i] if self.past[i] is not None else x.new_zeros(n - 1, x.shape[1])
        rows = torch.cat([past, x])
        self.past[i] = rows[-(n - 1):].clone()
        return sum(rows[j:j + x.shape[0]] * taps[:, j] for j in range(n))

    def _short_conv(self, i, n):
        b = f"blk.{i}.shortconv."
        B, C, x = self._linear(n, b + "in_proj").chunk(3, -1)
        return self._linear(C * self._taps(i, B * x, self.w[b + "conv.weight"].reshape(-1, 3)), b + "out_proj")

    def _mamba(self, i, n):
        b, S = f"blk.{i}.", 128
        silu = torch.nn.functional.silu
        inner = self.w[b + "ssm_out.weight"].shape[1]
        nh = inner // 32
        z, xbc, dt = self._linear(n, b + "ssm_in").split([inner, inner + 2 * S, nh], -1)
        xbc = silu(self._taps(i, xbc, self.w[b + "ssm_conv1d.weight"].reshape(-1, 4)) + self.w[b + "ssm_conv1d.bias"])
        x, B, C = xbc[:, :inner].reshape(-1, nh, 32), xbc[:, inner:inner + S], xbc[:, inner + S:]
        dt = torch.nn.functional.softplus(dt + self.w[b + "ssm_dt.bias"], threshold=50.0)
        decay = torch.exp(dt * self.w[b + "ssm_a"].reshape(-1))
        h = self.state[i] if self.state[i] is not None else x.new_zeros(nh, 32, S)
        y = torch.empty_like(x)
        for t in range(x.shape[0]):
            h = h * decay[t][:, None, None] + (dt[t][:, None] * x[t])[:, :, None] * B[t]
            y[t] = h @ C[t]
        self.state[i] = h
        y = (y + self.w[b + "ssm_d"].reshape(-1, 1) * x).reshape(-1, inner) * silu(z)
        return self._linear(self._norm(y, b + "ssm_norm"), b + "ssm_out")

    def _layer(self, i, x):
        b, gpt, gemma = f"blk.{i}.", self.arch == "gpt2", self.arch == "gemma3"
        scale = 0.246 if self.arch == "granitehybrid" else 1.0
        n = self._norm(x, b + "attn_norm")
        if b + "shortconv.conv.weight" in self.w:
            o = self._short_conv(i, n)
        elif b + "ssm_in.weight" in self.w:
            o = self._mamba(i, n)
        else:
            o = self._attention(i, n)
        if gemma:
            x = torch.clamp(x + self._norm(o, b + "post_attention_norm"), -65000, 65000)
        else:
            x = x + scale * o
        if gpt:
            x = torch.clamp(x, -10000, 10000)
        n = self._norm(x, b + "ffn_norm")
        up = self._linear(n, b + "ffn_up")
        if gpt:
            return torch.clamp(x + self._linear(self._gelu(up), b + "ffn_down"), -10000, 10000)
        gate = self._linear(n, b + "ffn_gate")
        d = self._linear((self._gelu(gate) if gemma else torch.nn.functional.silu(gate)) * up, b + "ffn_down")
        if gemma:
            return torch.clamp(x + self._norm(d, b + "post_ffw_norm"), -65000, 65000)
        return x + scale * d

    # -- rows of tokens -> logits after the last one
    def logits(self, tokens):
        for at in range(0, len(tokens), self.CHUNK):
            ids = torch.tensor(tokens[at:at + self.CHUNK], device=_device())
            x = self.w["token_embd.weight"][ids]
            if self.arch == "gpt2":
                x = x + self.w["position_embd.weight"][self.pos:self.pos + len(ids)]
            x = x * {"gemma3": self.spec.hidden ** 0.5, "granitehybrid": 12.0}.get(self.arch, 1.0)
            for i in range(self.spec.layers):
                x = self._layer(i, x)
            self.pos += len(ids)
        last = self._norm(x[-1:], "token_embd_norm" if self.arch == "lfm2" else "output_norm")[0]
        head = self.w.get("output.weight", self.w["token_embd.weight"])
        return (head @ last) / (3.0 if self.arch == "granitehybrid" else 1.0)


_exact: dict = {}


def _mix64(z):
    z &= (1 << 64) - 1
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & ((1 << 64) - 1)
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & ((1 << 64) - 1)
    return z ^ (z >> 31)


def _pick(logits, sample, seed, pos):
    """The next id: the first maximum, or the candidate sampler over each 256 ids' maximum."""
    if not sample:
        return int(torch.argmax(logits))
    pad = torch.nn.functional.pad(logits, (0, -logits.numel() % 256), value=float("-inf")).view(-1, 256)
    best, where = pad.max(1)
    order = torch.argsort(best, descending=True)[: SAMPLING["top_k"]].cpu()
    p = torch.exp((best.cpu()[order] - best.cpu()[order][0]) / SAMPLING["temperature"])
    u = (_mix64(seed + 0x9E3779B97F4A7C15 * (pos + 1)) >> 11) * 2.0 ** -53
    at = min(int(torch.searchsorted(torch.cumsum(p, 0), u * float(p.sum()))), len(order) - 1)
    return int(order[at]) * 256 + int(where[order[at]])


def exact(case, seed):
    key = (case["model"], case["kv"])
    if key not in _exact:
        _exact.clear()
        _exact[key] = _Exact(*key)
    m = _exact[key]
    prompts, forced = _tokens(case, seed)
    if case["kind"] == "batch":
        rows = []
        for s, prompt in enumerate(prompts):
            m.reset()
            rows.append(m.logits(prompt + [step[s] for step in forced]).cpu().numpy())
        return {"logits": np.stack(rows)}
    m.reset()
    if case["kind"] == "guided":
        return {"logits": m.logits(prompts[0] + [step[0] for step in forced[: case["new"] - 1]]).cpu().numpy()}
    w = WORKLOADS[case["model"]]
    y, ids = m.logits(prompts[0]), []
    while True:
        ids.append(_pick(y, case["sample"], int(seed), m.pos - 1))
        # the GPT-2, LFM2 and Granite loops also run the last id
        last, more = len(ids) == case["new"], w.spec.arch in ("gpt2", "lfm2", "granitehybrid")
        if ids[-1] in w.eos_ids or (last and not more):
            break
        y = m.logits(ids[-1:])
        if last:
            break
    return {"ids": None, "logits": y.cpu().numpy()}
