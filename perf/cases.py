"""Performance cases of the decode/prefill backend: what a program that uses it has it do, over the sizes it meets.

Kinds of case:
* ``decode``: one ``run_decode_batch`` step of a cut model (a few layers of the Llama-3-8B or Qwen2-7B shapes, block
  weights) over sessions that hold a context; the scheduler's inner loop.  Returns the logits and the KV pools that
  the step appended to.
* ``prompt``: one ``run_prefill_batch`` of a cut model, prompts of equal or of different lengths.  Returns the logits.
* ``tiny``: the same two calls on the float32 tiny model (dense weights, float32 KV pages), the smallest calls there
  are.
* ``extend``: the causal attention of new tokens over a paged context (a prompt, or a chunk that continues one).
* ``attend``: the decode attention of one token per sequence over paged contexts of different lengths.
* ``mlp``: a SwiGLU block with its residual and the next RMSNorm, in each quantized weight format, at any row count.

Sizes are fixed by the case alone; values (ids, weights, K/V, page placement) come from the seed.
"""
from __future__ import annotations

import math
import random
import zlib

import numpy as np
import torch

from cacheir_amd import compile_config, create_runtime, kernels
from cacheir_amd.artifact import ModelConfig
from cacheir_amd.weights import GGML_Q4_0, GGML_Q8_0, SyntheticQuant

PAGE = 16
VOCAB = 16384  # cut with the layers, so that the head keeps about the share of a step that it has in the whole model
MODELS = {
    # hidden, ffn, heads, kv heads, rope theta, eps
    "llama3-8b": (4096, 14336, 32, 8, 500000.0, 1e-5),
    "qwen2-7b": (3584, 18944, 28, 4, 1000000.0, 1e-6),
    "tiny": (256, 688, 4, 2, 10000.0, 1e-5),
}
WEIGHT_BYTES = {"q4_0": 18 / 32, "q8_0": 34 / 32, "int4": 0.5, "int8": 1.0, "f32": 4.0}


# ------------------------------------------------------------------ cases ------
def listed() -> list[dict]:
    return [
        # the first token of a request on the float32 tiny model (the reference's own artifact): launches and latency
        dict(name="tiny decode b1", kind="tiny", batch=1, tokens=33, step="decode"),
        # its prompt
        dict(name="tiny prompt 48", kind="tiny", batch=1, tokens=48, step="prompt"),
        # one user waiting for the next token
        dict(name="decode q4_0 b1", kind="decode", model="llama3-8b", quant="q4_0", layers=4, batch=1, lo=2047, hi=2047,
             prefix=0),
        # a few users with contexts of their own lengths
        dict(name="decode q4_0 b8", kind="decode", model="llama3-8b", quant="q4_0", layers=4, batch=8, lo=300, hi=1500,
             prefix=0),
        # the headline decode step: 32 sequences at 2048 tokens
        dict(name="decode q4_0 b32", kind="decode", model="llama3-8b", quant="q4_0", layers=4, batch=32, lo=2047,
             hi=2047, prefix=0),
        # a full server: 128 sequences behind one shared 1024-token prefix, ragged suffixes
        dict(name="decode q8_0 b128 prefix", kind="decode", model="qwen2-7b", quant="q8_0", layers=2, batch=128, lo=64,
             hi=7168, prefix=1024),
        # one long prompt
        dict(name="prompt q4_0 2048", kind="prompt", model="llama3-8b", quant="q4_0", layers=2, batch=1, lo=2048,
             hi=2048),
        # several short prompts of odd lengths admitted together
        dict(name="prompt q8_0 5 ragged", kind="prompt", model="qwen2-7b", quant="q8_0", layers=2, batch=5, lo=37,
             hi=301),
        # a chunk of a long prompt over the context before it
        dict(name="extend 2x509 past 3500", kind="extend", heads=28, kv_heads=4, batch=2, q_len=509, past=3500),
        # decode attention of 64 sequences between 512 and 4096 tokens, pages anywhere in the pool
        dict(name="attend b64 ragged", kind="attend", heads=32, kv_heads=8, batch=64, lo=512, hi=4096),
        # the MLP of a full server's step
        dict(name="mlp q8_0 m128", kind="mlp", model="qwen2-7b", quant="q8_0", m=128),
        # the MLP of row-quantized (AWQ-style int4) weights at an odd row count
        dict(name="mlp int4 m77", kind="mlp", model="llama3-8b", quant="int4", m=77),
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["tiny", "decode", "decode", "prompt", "prompt", "extend", "attend", "mlp", "mlp", "mlp"])
    if kind == "tiny":
        return dict(kind=kind, batch=rng.randint(1, 4), tokens=_log(rng, 3, 96), step=rng.choice(["decode", "prompt"]))
    if kind == "decode":
        model, quant, layers = rng.choice([("llama3-8b", "q4_0", 4), ("llama3-8b", "q8_0", 2), ("qwen2-7b", "q8_0", 2),
                                           ("qwen2-7b", "q4_0", 3)])
        batch, hi = _log(rng, 1, 128), _log(rng, 96, 8000)
        hi = min(hi, 500000 // batch)
        lo = max(32, int(hi * rng.uniform(0.1, 1.0)))
        return dict(kind=kind, model=model, quant=quant, layers=layers, batch=batch, lo=lo, hi=max(lo, hi),
                    prefix=rng.choice([0, 0, 128, 1024]))
    if kind == "prompt":
        model, quant, layers = rng.choice([("llama3-8b", "q4_0", 2), ("llama3-8b", "q8_0", 1), ("qwen2-7b", "q8_0", 1),
                                           ("qwen2-7b", "q4_0", 2)])
        batch = rng.choice([1, 1, 2, 3, 4, 7])
        hi = _log(rng, 9, 2040 // batch)
        return dict(kind=kind, model=model, quant=quant, layers=layers, batch=batch,
                    lo=hi if rng.random() < 0.5 else max(3, int(hi * rng.uniform(0.3, 1.0))), hi=hi)
    if kind == "extend":
        heads, kv_heads = rng.choice([(32, 8), (28, 4), (16, 8), (8, 8)])
        batch = _log(rng, 1, 8)
        q_len = _log(rng, 5, 2048 // batch)
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, batch=batch, q_len=q_len,
                    past=rng.choice([0, rng.randint(1, 500), rng.randint(500, 6000)]))
    if kind == "attend":
        heads, kv_heads = rng.choice([(32, 8), (28, 4), (16, 8), (8, 8)])
        batch, hi = _log(rng, 1, 128), _log(rng, 100, 8000)
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, batch=batch, lo=max(16, int(hi * rng.uniform(0.1, 1.0))),
                    hi=hi)
    return dict(kind=kind, model=rng.choice(["llama3-8b", "qwen2-7b"]),
                quant=rng.choice(["q4_0", "q4_0", "q8_0", "int4", "int8"]), m=_log(rng, 1, 2048))


def _lengths(case: dict) -> list[int]:
    """Token counts per sequence, spread evenly between lo and hi in an order of their own (fixed by the case)."""
    b, lo, hi = case["batch"], case["lo"], case["hi"]
    lens = [hi if b == 1 else lo + (hi - lo) * i // (b - 1) for i in range(b)]
    random.Random(b * 1000003 + lo * 1009 + hi).shuffle(lens)
    return lens


# ------------------------------------------------------------------ values -----
def _gen(seed: int, *what) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 2654435761 + zlib.crc32(repr(what).encode())) & 0x7FFFFFFFFFFF)
    return g


def _randn(shape, seed: int, *what, dtype=torch.float32) -> torch.Tensor:
    return torch.randn(shape, generator=_gen(seed, *what), device="cuda", dtype=torch.float32).to(dtype)


def _blocks(quant: str, n: int, k: int, seed: int, *what) -> tuple[torch.Tensor, torch.Tensor]:
    """N(0, 0.02) weights in blocks of 32: fp16 scales [n, k/32] and codes [n, k/32, 32], value = scale * code."""
    w = _randn((n, k // 32, 32), seed, quant, *what) * 0.02
    if quant == "q4_0":
        big = w.gather(2, w.abs().argmax(dim=2, keepdim=True))
        d = big / -8.0
        q = torch.floor(w / d + 8.5).clamp_(0, 15) - 8
    else:
        d = w.abs().amax(dim=2, keepdim=True) / 127.0
        q = torch.round(w / d).clamp_(-127, 127)
    return d.squeeze(2).half(), q.to(torch.int8)


def _gguf(quant: str, d: torch.Tensor, q: torch.Tensor) -> torch.Tensor:
    """GGUF bytes [n, row_bytes] of the blocks."""
    n, nb = d.shape
    if quant == "q4_0":
        c = (q + 8).view(torch.uint8)
        body = c[:, :, :16] | (c[:, :, 16:] << 4)
    else:
        body = q.view(torch.uint8)
    return torch.cat([d.view(torch.uint8).view(n, nb, 2), body], dim=2).reshape(n, -1)


def _rows(bits: int, n: int, k: int, seed: int, *what) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """N(0, 0.02) weights with a scale and a zero point per row: codes uint8 [n, k], scales fp32, zero points int32."""
    w = _randn((n, k), seed, bits, *what) * 0.02
    lo, hi = w.amin(dim=1), w.amax(dim=1)
    s = (hi - lo) / ((1 << bits) - 1)
    z = torch.round(-lo / s).to(torch.int32)
    q = torch.round(w / s[:, None] + z[:, None]).clamp_(0, (1 << bits) - 1).to(torch.uint8)
    return q, s, z


class _DrawnWeights(SyntheticQuant):
    """Weights drawn per key, so that a second reader of the same seed finds the same ones in any order."""

    def __init__(self, quant: str, seed: int):
        super().__init__(GGML_Q4_0 if quant == "q4_0" else GGML_Q8_0, "cuda", seed=seed)
        self.quant, self.seed = quant, seed

    def blocks_device(self, key):
        n, k = self.shapes[key]
        return _gguf(self.quant, *_blocks(self.quant, n, k, self.seed, key)).reshape(-1), self.fmt, n, k

    def dense_device(self, key, dtype):
        return _dense(key, self.shapes[key], self.seed).to(dtype)


class _DenseWeights:
    """The float32 tiny model's weights, as arrays."""

    def __init__(self, shapes: dict, seed: int):
        self._w = {k: _dense(k, s, seed).cpu().numpy() for k, s in shapes.items()}

    def has_blocks(self, key):
        return False

    def dense(self, key):
        return self._w[key]


def _dense(key: str, shape, seed: int) -> torch.Tensor:
    """Norm gains around one, embeddings N(0, 0.1), other matrices N(0, 1 / k), in values that fp16 holds too."""
    w = _randn(tuple(shape), seed, key)
    w = 1.0 + 0.1 * w if len(shape) == 1 else w * (0.1 if "embed" in key else shape[1] ** -0.5)
    return w.half().float()


def _context(case: dict, seed: int, layer: int, row: int | str, tokens: int) -> tuple[torch.Tensor, torch.Tensor]:
    """K and V of a row's cached tokens ([tokens, kv heads, head dim]); row "prefix" is the shared part."""
    hidden, _, heads, kvh, _, _ = MODELS[case.get("model", "tiny")]
    dt = torch.float32 if case["kind"] == "tiny" else torch.float16
    kv = _randn((2, tokens, kvh, hidden // heads), seed, "kv", layer, row, dtype=dt)
    return kv[0], kv[1]


# ------------------------------------------------------------------ prepare ----
def _config(case: dict) -> ModelConfig:
    name = case.get("model", "tiny")
    h, f, heads, kvh, theta, eps = MODELS[name]
    tiny = name == "tiny"
    return ModelConfig(architecture=f"{name}-shape", hidden_size=h, intermediate_size=f,
                       num_layers=2 if tiny else case["layers"], num_attention_heads=heads, num_key_value_heads=kvh,
                       vocab_size=1024 if tiny else VOCAB, max_position_embeddings=16384, rope_theta=theta,
                       rms_norm_eps=eps, dtype="float32" if tiny else "float16")


def _ids(case: dict, seed: int, lens: list[int]) -> list[list[int]]:
    rng = np.random.default_rng(seed)
    return [rng.integers(0, _config(case).vocab_size, n).tolist() for n in lens]


def _runtime(case: dict, seed: int, pages: int):
    cfg = _config(case)
    if case["kind"] == "tiny":
        art = compile_config(cfg)
        src = _DenseWeights({s.key: tuple(s.tensor_type.shape) for s in art.graph("decode").weights.values()}, seed)
    else:
        art = compile_config(cfg, quant=case["quant"])
        src = _DrawnWeights(case["quant"], seed)
    return create_runtime(art, backend="rocm", source=src, kv_capacity_pages=pages)


def _fill(cache, layer: int, first_page: int, k: torch.Tensor, v: torch.Tensor) -> None:
    """Write a row's tokens into its pages from page ``first_page`` on."""
    n = k.shape[0]
    pages = -(-n // PAGE)
    slots = torch.tensor(cache.slots[first_page:first_page + pages], device="cuda")
    for pool, x in zip(cache.allocator.layer_pools(layer), (k, v)):
        pad = torch.zeros((pages * PAGE - n, *x.shape[1:]), dtype=x.dtype, device=x.device)
        pool[slots] = torch.cat([x, pad]).view(pages, PAGE, *x.shape[1:]).transpose(1, 2)


def _decode_state(case: dict, seed: int, lens: list[int], prefix: int) -> dict:
    pages = prefix // PAGE + sum(-(-(n + 1) // PAGE) for n in lens) + 33 * 4
    base = _runtime(case, seed, pages)
    layers = base.config.num_layers
    if prefix:
        base.kv_cache.ensure_capacity(prefix)
        base.kv_cache.tokens = prefix
        for layer in range(layers):
            _fill(base.kv_cache, layer, 0, *_context(case, seed, layer, "prefix", prefix))
    sessions = []
    for row, n in enumerate(lens):
        s = base.fork()
        if prefix:
            s.kv_cache.alias_prefix(base.kv_cache.slots, prefix)
        s.kv_cache.ensure_capacity(prefix + n + 1)
        s.kv_cache.tokens = prefix + n
        for layer in range(layers):
            _fill(s.kv_cache, layer, prefix // PAGE, *_context(case, seed, layer, row, n))
        sessions.append(s)
    return dict(kind="decode", base=base, sessions=sessions, ids=[i[0] for i in _ids(case, seed, [1] * len(lens))])


def _paged(case: dict, seed: int, lens: list[int]) -> dict:
    """K/V pools of the rows' contexts with their pages placed at random, the page table and the lengths."""
    kvh, d = case["kv_heads"], 128
    npg = [-(-n // PAGE) for n in lens]
    slots = sum(npg)
    kv = _randn((2, slots, kvh, PAGE, d), seed, "pool", dtype=torch.float16)
    perm = np.random.default_rng(seed).permutation(slots).astype(np.int32)
    table, at = np.zeros((len(lens), max(npg)), np.int32), 0
    for b, p in enumerate(npg):
        table[b, :p] = perm[at:at + p]
        at += p
    return dict(k=kv[0], v=kv[1], table=torch.from_numpy(table).cuda(),
                lens=torch.tensor(lens, dtype=torch.int32, device="cuda"))


def _attention_inputs(case: dict, seed: int) -> dict:
    b = case["batch"]
    q_len = case.get("q_len", 1)
    lens = [case["past"] + q_len] * b if case["kind"] == "extend" else _lengths(case)
    st = _paged(case, seed, lens)
    st["q"] = _randn((b * q_len, case["heads"], 128), seed, "q", dtype=torch.float16)
    return st


def _mlp_inputs(case: dict, seed: int) -> dict:
    h, _, _, _, _, eps = MODELS[case["model"]]
    m = case["m"]
    x = _randn((m, h), seed, "x")
    outliers = torch.randperm(h, generator=_gen(seed, "outliers"), device="cuda")[:16]
    x[:, outliers] *= 8.0  # the few large channels of a normed stream
    return dict(x=x.half(), resid=_randn((m, h), seed, "resid"), gain=(1.0 + 0.1 * _randn((h,), seed, "gain")).half(),
                eps=eps)


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "decode":
        return _decode_state(case, seed, _lengths(case), case["prefix"])
    if kind == "tiny" and case["step"] == "decode":
        return _decode_state(case, seed, [case["tokens"]] * case["batch"], 0)
    if kind in ("prompt", "tiny"):
        lens = _lengths(case) if kind == "prompt" else [case["tokens"]] * case["batch"]
        base = _runtime(case, seed, sum(-(-n // PAGE) for n in lens) + 33 * 4)
        return dict(kind="prompt", base=base, sessions=[base.fork() for _ in lens], ids=_ids(case, seed, lens))
    if kind in ("extend", "attend"):
        st = _attention_inputs(case, seed)
        rows, context = st["q"].shape[0], st["table"].shape[1] * PAGE
        st["ws"] = kernels.attention_workspace(rows, case["heads"], 128, context, "cuda")
        return dict(st, kind=kind, q_len=case.get("q_len", 1))
    st = _mlp_inputs(case, seed)
    h, f = MODELS[case["model"]][:2]
    quant = case["quant"]
    if quant in ("q4_0", "q8_0"):
        gate, up, down = (_gguf(quant, *_blocks(quant, n, k, seed, w))
                          for w, n, k in (("gate", f, h), ("up", f, h), ("down", h, f)))
        fmt = kernels.FMT_NAMES[quant]
        st["gate_up"] = kernels.QWeight.from_blocks(kernels.interleave_gate_up(gate, up, f).reshape(-1), fmt, 2 * f, h)
        st["down"] = kernels.QWeight.from_blocks(down.reshape(-1), fmt, h, f)
    else:
        bits = int(quant[3:])
        pack = (lambda q: q[:, 0::2] | (q[:, 1::2] << 4)) if bits == 4 else (lambda q: q)
        (gq, gs, gz), (uq, us, uz) = _rows(bits, f, h, seed, "gate"), _rows(bits, f, h, seed, "up")
        pair = lambda a, b: torch.stack([a.view(f // 16, 16), b.view(f // 16, 16)], dim=1).reshape(-1)
        st["gate_up"] = kernels.QWeight.from_rows(kernels.interleave_gate_up(pack(gq), pack(uq), f), pair(gs, us),
                                                  pair(gz, uz), bits, 2 * f, h)
        dq, ds, dz = _rows(bits, h, f, seed, "down")
        st["down"] = kernels.QWeight.from_rows(pack(dq).contiguous(), ds, dz, bits, h, f)
    return dict(st, kind=kind, h=torch.empty_like(st["resid"]), xn=torch.empty_like(st["x"]))


# ------------------------------------------------------------------ run --------
def run(state: dict):
    kind = state["kind"]
    if kind == "decode":
        logits = state["base"].run_decode_batch(state["sessions"], state["ids"])
        for s in state["sessions"]:  # the next pass decodes the same token again
            s.kv_cache.tokens -= 1
        pool = state["base"].kv_allocator
        return {"logits": logits, "k": pool.k, "v": pool.v}
    if kind == "prompt":
        return state["base"].run_prefill_batch(state["sessions"], state["ids"])
    if kind == "extend":
        return kernels.paged_prefill_attention(state["q"], state["k"], state["v"], state["table"], state["lens"],
                                               state["q_len"], workspace=state["ws"])
    if kind == "attend":
        return kernels.paged_decode_attention(state["q"], state["k"], state["v"], state["table"], state["lens"],
                                              workspace=state["ws"])
    act = kernels.qgemm_swiglu(state["x"], state["gate_up"])
    part = kernels.qgemm_partial(act, state["down"])
    h, xn = kernels.epilogue_residual_rmsnorm(part, state["resid"], state["gain"], state["eps"], state["h"],
                                              state["xn"])
    return {"act": act, "h": h, "xn": xn}


# ------------------------------------------------------------------ work -------
def _model_work(case: dict, lens: list[int], past: list[int], shared: int) -> dict:
    """Weights once, the context's K/V once (a shared prefix once), new K/V and logits written once."""
    cfg = _config(case)
    h, f, d = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    kvh, heads = cfg.num_key_value_heads, cfg.num_attention_heads
    per_layer = 2 * h * h + 2 * h * kvh * d + 3 * h * f
    rows = sum(lens)
    kv_elt = 4 if case["kind"] == "tiny" else 2
    wb = WEIGHT_BYTES["f32" if case["kind"] == "tiny" else case["quant"]]
    kv_tokens = shared + sum(p - shared for p in past) + rows
    seen = sum(n * p + n * (n + 1) // 2 for n, p in zip(lens, past))  # (query, key) pairs under the causal mask
    params = cfg.num_layers * per_layer + cfg.vocab_size * h
    return {"bytes": wb * params + cfg.num_layers * kv_tokens * 2 * kvh * d * kv_elt + 4 * rows * cfg.vocab_size,
            "flops": 2 * rows * params + cfg.num_layers * 4 * heads * d * seen}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "decode":
        lens = _lengths(case)
        return _model_work(case, [1] * len(lens), [case["prefix"] + n for n in lens], case["prefix"])
    if kind == "tiny":
        b, t = case["batch"], case["tokens"]
        new, past = (1, t) if case["step"] == "decode" else (t, 0)
        return _model_work(case, [new] * b, [past] * b, 0)
    if kind == "prompt":
        lens = _lengths(case)
        return _model_work(case, lens, [0] * len(lens), 0)
    if kind in ("extend", "attend"):
        b, q = case["batch"], case.get("q_len", 1)
        lens = [case["past"] + q] * b if kind == "extend" else _lengths(case)
        seen = sum(q * (n - q) + q * (q + 1) // 2 for n in lens)
        return {"bytes": 4 * sum(lens) * case["kv_heads"] * 128 + 4 * b * q * case["heads"] * 128,
                "flops": 4 * case["heads"] * 128 * seen}
    h, f = MODELS[case["model"]][:2]
    m = case["m"]
    return {"bytes": 3 * h * f * WEIGHT_BYTES[case["quant"]] + m * (2 * h + 2 * f + 4 * h + 4 * h + 2 * h),
            "flops": 6 * m * h * f}


# ------------------------------------------------------------------ exact ------
def _rms64(x: torch.Tensor, gain: torch.Tensor, eps: float) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + eps) * gain.double()


def _attend64(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """q [n, heads, d] are the last n of the t tokens k, v [t, kv heads, d] hold; causal."""
    n, heads, d = q.shape
    t, kvh = k.shape[:2]
    out = torch.empty_like(q)
    ahead = torch.arange(t, device=q.device)[None, :] > torch.arange(t - n, t, device=q.device)[:, None]
    for g in range(kvh):
        for j in range(heads // kvh):
            i = g * (heads // kvh) + j
            s = (q[:, i] @ k[:, g].T) * d ** -0.5
            out[:, i] = torch.softmax(s.masked_fill(ahead, -math.inf), dim=-1) @ v[:, g]
    return out


def _rope64(x: torch.Tensor, pos: torch.Tensor, theta: float) -> torch.Tensor:
    """Rotation of the pairs (2i, 2i + 1); the inverse frequencies are those of the model, in 32 bits."""
    d = x.shape[-1]
    inv = (1.0 / (theta ** (np.arange(0, d // 2, dtype=np.float32) * 2.0 / d))).astype(np.float32)
    a = (pos.double()[:, None] * torch.from_numpy(inv).to(x.device).double())[:, None, :]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * a.cos() - x1 * a.sin(), x0 * a.sin() + x1 * a.cos()], dim=-1).flatten(-2)


def _forward64(case: dict, seed: int, ids: list[list[int]], past: list[int], prefix: int) -> list[torch.Tensor]:
    """Logits of every row's new tokens, the row's cached context (if any) before them."""
    cfg = _config(case)
    h, f, d = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    heads, kvh = cfg.num_attention_heads, cfg.num_key_value_heads

    def mat(key: str, n: int, k: int) -> torch.Tensor:
        if case["kind"] == "tiny":
            return _dense(key, (n, k), seed).double()
        s, q = _blocks(case["quant"], n, k, seed, key)
        return (s.double()[:, :, None] * q).view(n, k)

    def gain(key: str) -> torch.Tensor:
        return _dense(key, (h,), seed)

    sizes = [len(i) for i in ids]
    pos = torch.cat([torch.arange(p, p + n, device="cuda") for p, n in zip(past, sizes)])
    embed = _dense("model.embed_tokens.weight", (cfg.vocab_size, h), seed)
    x = embed[torch.tensor(sum(ids, []), device="cuda")].double()
    for layer in range(cfg.num_layers):
        p = f"model.layers.{layer}"
        y = _rms64(x, gain(f"{p}.input_layernorm.weight"), cfg.rms_norm_eps)
        q, k, v = (y @ mat(f"{p}.self_attn.{w}_proj.weight", n * d, h).T
                   for w, n in (("q", heads), ("k", kvh), ("v", kvh)))
        q = _rope64(q.view(-1, heads, d), pos, cfg.rope_theta)
        k = _rope64(k.view(-1, kvh, d), pos, cfg.rope_theta)
        v = v.view(-1, kvh, d)
        outs, at = [], 0
        shared = _context(case, seed, layer, "prefix", prefix) if prefix else None
        for row, n in enumerate(sizes):
            kk, vv = [k[at:at + n]], [v[at:at + n]]
            if past[row]:
                ck, cv = _context(case, seed, layer, row, past[row] - prefix)
                kk, vv = [ck.double()] + kk, [cv.double()] + vv
                if prefix:
                    kk, vv = [shared[0].double()] + kk, [shared[1].double()] + vv
            outs.append(_attend64(q[at:at + n], torch.cat(kk), torch.cat(vv)))
            at += n
        x = x + torch.cat(outs).reshape(-1, heads * d) @ mat(f"{p}.self_attn.o_proj.weight", h, heads * d).T
        y = _rms64(x, gain(f"{p}.post_attention_layernorm.weight"), cfg.rms_norm_eps)
        gate, up = (y @ mat(f"{p}.mlp.{w}_proj.weight", f, h).T for w in ("gate", "up"))
        y = torch.nn.functional.silu(gate) * up
        x = x + y @ mat(f"{p}.mlp.down_proj.weight", h, f).T
    logits = _rms64(x, gain("model.norm.weight"), cfg.rms_norm_eps) @ mat("lm_head.weight", cfg.vocab_size, h).T
    return list(logits.split(sizes))


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "decode" or (kind == "tiny" and case["step"] == "decode"):
        lens = _lengths(case) if kind == "decode" else [case["tokens"]] * case["batch"]
        prefix = case.get("prefix", 0)
        rows = _forward64(case, seed, _ids(case, seed, [1] * len(lens)), [prefix + n for n in lens], prefix)
        return {"logits": torch.stack(rows), "k": None, "v": None}
    if kind in ("prompt", "tiny"):
        lens = _lengths(case) if kind == "prompt" else [case["tokens"]] * case["batch"]
        rows = _forward64(case, seed, _ids(case, seed, lens), [0] * len(lens), 0)
        return torch.nn.utils.rnn.pad_sequence(rows, batch_first=True)  # zeros past a prompt's end
    if kind in ("extend", "attend"):
        st = _attention_inputs(case, seed)
        n, outs = case.get("q_len", 1), []
        for b, t in enumerate(st["lens"].tolist()):
            pages = st["table"][b, : -(-t // PAGE)].long()
            k, v = (p[pages].transpose(1, 2).reshape(-1, case["kv_heads"], 128)[:t].double()
                    for p in (st["k"], st["v"]))
            outs.append(_attend64(st["q"][b * n:(b + 1) * n].double(), k, v))
        return torch.cat(outs)
    st = _mlp_inputs(case, seed)
    h, f = MODELS[case["model"]][:2]
    quant = case["quant"]

    def mat(what: str, n: int, k: int) -> torch.Tensor:
        if quant in ("q4_0", "q8_0"):
            s, q = _blocks(quant, n, k, seed, what)
            return (s.double()[:, :, None] * q).view(n, k)
        q, s, z = _rows(int(quant[3:]), n, k, seed, what)
        return (q.double() - z.double()[:, None]) * s.double()[:, None]

    x = st["x"].double()
    act = torch.nn.functional.silu(x @ mat("gate", f, h).T) * (x @ mat("up", f, h).T)
    out = st["resid"].double() + act @ mat("down", h, f).T
    return {"act": act, "h": out, "xn": _rms64(out, st["gain"], st["eps"])}


# ------------------------------------------------------------------ tolerance --
def tolerance(case: dict) -> dict:
    """About four times what the paths are measured off ``exact`` (in brackets)."""
    kind = case["kind"]
    if kind == "tiny":  # 32-bit sums through two layers (4.9e-7)
        return {"rel": 2e-6}
    if kind in ("decode", "prompt"):  # 16-bit GEMM inputs, q, K and V through a few layers (1.3e-3)
        return {"rel": 5e-3}
    return {"rel": 1.2e-3}  # 16-bit probabilities and results; 16-bit activations between two products (2.9e-4)
