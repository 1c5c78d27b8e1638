"""The work whose time is followed, as cases: what a serving program has this framework do.

Sizes are those of the benchmark's workloads (decode at batch 32, the mixed chunked-prefill step, the large pool,
speculative verify, the attention block, whole-model steps) and of the tests, at the two model shapes both use:
hidden 1024 with a 3072-wide MLP and hidden 2048 with a 6144-wide one, 16 query and 8 kv heads of 128, pages of
16 tokens. Listed sizes are deliberately not all round; ``draw`` spreads over the whole range.

Kinds of case:

  step     PagedKv.plan, then PagedKv.layer for each layer: the engine's attention step (append + attention) for any
           mix of decode, verify and prefill tokens. Outputs: each layer's attention output and its K and V pools.
  block    PagedKv.plan, then PagedKv.attention_block for each layer: norm, qkv projection, append + attention,
           output projection into the residual. Outputs: the residual, and each layer's pools.
  mlp      rmsnorm_rows, the gate/up projection with silu_mul, the down projection into the residual.
  sample   the device sampler and the drafted tokens' probabilities over rows of logits (C ABI).
  backend  Backend.forward over a model directory, Backend.sample, and the logits: a prompt, or one decode step over
           cached prompts.
"""
from __future__ import annotations

import ctypes
import functools
import json
import math
import os
import random
import tempfile

import numpy as np
import torch

from ember_amd import _lib
from ember_amd import kernels as K
from ember_amd.backend import BackendOptions, SampleRequest, SamplingParams, create_backend
from ember_amd.paged_kv import PagedKv, StepBatch

PAGE, D = 16, 128
THETA, EPS = 1e6, 1e-6
VOCAB = 151936
SHAPES = {"0.6B": (1024, 3072), "1.7B": (2048, 6144)}  # hidden, MLP width

STEP = dict(kind="step", seqs=1, new=1, chunks=0, chunk=0, ctx_lo=256, ctx_hi=4096, log=False, prefix=0, layers=1,
            heads=16, kv_heads=8, dtype="f16", lens=1)


def _step(name: str, **kw) -> dict:
    return {"name": name, **STEP, **kw}


def listed() -> list:
    return [
        # One user's chat turn: a single sequence's decode, a few pages of context. All latency.
        _step("decode_b1", seqs=1, ctx_lo=640, ctx_hi=640, layers=4),
        # Batched decode, the headline workload: 32 sequences of 256 to 4096 tokens.
        _step("decode_b32", seqs=32, ctx_lo=256, ctx_hi=4096, layers=4, lens=2),
        # A full card's decode: 256 sequences, long and short (log-uniform 512 to 16384), from a large pool.
        _step("decode_b256_long", seqs=256, ctx_lo=512, ctx_hi=16384, log=True, layers=2, lens=3),
        # Speculative verify: 64 sequences, 4 drafted tokens and one more each.
        _step("verify_b64", seqs=64, new=5, ctx_lo=512, ctx_hi=4096, layers=2, lens=4),
        # Continuous batching: 4 prompt chunks of 512 beside 60 decodes, all behind one shared 1024-token prefix.
        _step("mixed_b64", seqs=64, chunks=4, chunk=512, ctx_lo=1152, ctx_hi=3072, prefix=1024, layers=2, lens=5),
        # A first prompt: 500 tokens of one sequence, nothing cached.
        _step("prefill_500", seqs=1, chunks=1, chunk=500, ctx_lo=500, ctx_hi=500, layers=2),
        # A long document's last chunk, or the re-prefill of a preempted sequence: 2000 tokens on a 12,000 context.
        _step("prefill_long", seqs=1, chunks=1, chunk=2000, ctx_lo=14000, ctx_hi=14000, layers=1),
        # The attention half of a layer at batch 32, projections included.
        dict(name="block_b32", kind="block", model="1.7B", seqs=32, ctx_lo=256, ctx_hi=4096, layers=2, lens=6),
        # The MLP half of a layer for a step of 48 tokens (a wide decode batch or a short chunk).
        dict(name="mlp_b48", kind="mlp", model="1.7B", tokens=48, packed=True),
        # Sampling 16 rows of the full vocabulary with top-k and top-p, and the drafted tokens' probabilities.
        dict(name="sample_b16", kind="sample", rows=16, vocab=VOCAB, temperature=0.8, top_k=40, top_p=0.9, min_p=0.0),
        # A whole model's prompt, near the default batch limit: 1800 tokens to the first generated one.
        dict(name="model_prompt_1800", kind="backend", phase="prompt", seqs=1, tokens=1800),
        # A whole model's decode step, one user.
        dict(name="model_decode_b1", kind="backend", phase="decode", seqs=1, tokens=300),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choices(["decode", "verify", "mixed", "prefill", "block", "mlp", "sample", "prompt", "model_decode"],
                       [4, 2, 2, 4, 2, 3, 3, 2, 1])[0]
    lens = rng.randrange(10, 1 << 20)
    if kind in ("decode", "verify", "mixed", "prefill"):
        heads = rng.choice([16, 16, 16, 32, 40, 64])
        c = {**STEP, "heads": heads, "lens": lens, "layers": rng.choice([1, 2])}
        if kind == "prefill":
            chunks = rng.choice([1, 1, 2, 4])
            chunk = _log_int(rng, 16, 2048 // chunks)
            before = rng.choice([0, 0, _log_int(rng, 16, 12000 // chunks)])
            # heads x tokens x context kept within the largest listed chunk's
            while heads * chunks * chunk * (before + chunk) > 16 * 2000 * 14000:
                before //= 2
                chunk = max(16, chunk * 3 // 4)
            c.update(seqs=chunks, chunks=chunks, chunk=chunk, ctx_lo=chunk + before // 2, ctx_hi=chunk + before)
            if rng.random() < 0.1:  # f32 pages: the parity path, small
                c.update(seqs=1, chunks=1, chunk=min(chunk, 128), ctx_lo=300, ctx_hi=300, dtype="f32", heads=16)
            return c
        hi = _log_int(rng, 64, 16384)
        lo = max(17, hi // rng.choice([1, 2, 8, 32]))
        most = 256 if kind == "decode" else 64
        seqs = min(_log_int(rng, 1, most), max(1, 1_000_000 // hi))
        c.update(seqs=seqs, ctx_lo=lo, ctx_hi=max(lo, hi), log=rng.random() < 0.5)
        if kind == "verify":
            c.update(new=rng.randint(2, 8))
        elif kind == "mixed":
            chunk = _log_int(rng, 24, 512)
            c.update(seqs=seqs + 2, chunks=min(2, seqs), chunk=chunk, ctx_lo=chunk + 17, ctx_hi=max(chunk + 17, min(hi, 4096)),
                     heads=rng.choice([16, 32]))
        elif rng.random() < 0.1:
            c.update(dtype="f32", ctx_hi=max(lo, min(hi, 2048)), ctx_lo=min(lo, 2048), seqs=min(seqs, 32), heads=16)
        return c
    model = rng.choice(list(SHAPES))
    if kind == "block":
        hi = _log_int(rng, 64, 4096)
        return dict(kind="block", model=model, seqs=_log_int(rng, 1, 64), ctx_lo=max(17, hi // 8), ctx_hi=hi, layers=2, lens=lens)
    if kind == "mlp":
        return dict(kind="mlp", model=model, tokens=_log_int(rng, 1, 64), packed=rng.random() < 0.7)
    if kind == "sample":
        t, k, p, m = rng.choice([(0.0, 0, 1.0, 0.0), (1.0, 0, 1.0, 0.0), (0.6, 20, 0.95, 0.0), (0.8, 40, 0.9, 0.0),
                                 (1.0, 0, 0.95, 0.0), (1.2, 0, 1.0, 0.02), (0.7, 100, 0.8, 0.01), (0.9, 1000, 1.0, 0.0)])
        return dict(kind="sample", rows=_log_int(rng, 1, 64), vocab=rng.choice([8192, 32003, VOCAB, VOCAB]),
                    temperature=t, top_k=k, top_p=p, min_p=m)
    if kind == "prompt":
        seqs = rng.choice([1, 1, 2, 3])
        return dict(kind="backend", phase="prompt", seqs=seqs, tokens=_log_int(rng, 20, 1800 // seqs))
    return dict(kind="backend", phase="decode", seqs=_log_int(rng, 1, 8), tokens=_log_int(rng, 16, 500))


# ---- what a case holds: lengths and pages -------------------------------------------------------------


def _contexts(case: dict) -> list:
    """Each sequence's context after the step: fixed by the case, not by the seed, so the work is the case's."""
    rng = random.Random(case["lens"])
    lo, hi = case["ctx_lo"], case["ctx_hi"]
    one = (lambda: _log_int(rng, lo, hi)) if case.get("log") else (lambda: rng.randint(lo, hi))
    return [max(one(), case.get("prefix", 0) + n) for n in _new_tokens(case)]  # nobody writes into a shared prefix


def _new_tokens(case: dict) -> list:
    chunks = case.get("chunks", 0)
    return [case.get("chunk", 0)] * chunks + [case.get("new", 1)] * (case["seqs"] - chunks)


def _layout(case: dict, seed: int):
    """(contexts, new tokens, block tables [seqs, width], pool blocks): pages scattered over the pool."""
    ctx, new = _contexts(case), _new_tokens(case)
    prefix = case.get("prefix", 0) // PAGE
    pages = [(c + PAGE - 1) // PAGE for c in ctx]
    need = prefix + sum(p - prefix for p in pages)
    num_blocks = need + need // 8 + 8
    order = np.random.default_rng(seed).permutation(num_blocks).astype(np.int32)
    tables = np.zeros((len(ctx), max(pages)), np.int32)
    at = prefix
    for s, p in enumerate(pages):
        tables[s, :prefix] = order[:prefix]
        tables[s, prefix:p] = order[at:at + p - prefix]
        at += p - prefix
    return ctx, new, tables, num_blocks


def _batch(ctx, new, tables) -> StepBatch:
    pos = np.concatenate([np.arange(c - n, c) for c, n in zip(ctx, new)]).astype(np.int32)
    qs = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    return StepBatch(tokens=np.zeros(pos.size, np.int32), positions=pos, query_start=qs,
                     context_len=np.asarray(ctx, np.int32), block_tables=tables, max_blocks=int(tables.shape[1]))


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, scale=1.0, dtype=torch.float16) -> torch.Tensor:
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def _norm_weight(g, n: int) -> torch.Tensor:
    return 1 + 0.1 * torch.randn(n, generator=g, device="cuda")


class _Pool:
    """One layer's K or V pool as a device array that keeps its PagedKv alive (pool_view's tensors do not)."""

    def __init__(self, kv: PagedKv, layer: int, which: str):
        view = kv.pool_view(layer, which)
        self.kv = kv
        self.__cuda_array_interface__ = {"shape": tuple(view.shape), "typestr": "<f2" if view.dtype == torch.float16 else "<f4",
                                         "data": (view.data_ptr(), False), "version": 2, "strides": None}


def _pool(kv: PagedKv, layer: int, which: str) -> torch.Tensor:
    return torch.as_tensor(_Pool(kv, layer, which), device="cuda")


def _kv(case: dict, seed: int, heads: int, kv_heads: int, dtype=torch.float16):
    """A PagedKv with every page holding values as normed, rotated keys and values have them (unit scale)."""
    ctx, new, tables, num_blocks = _layout(case, seed)
    kv = PagedKv(n_layers=case["layers"], n_heads=heads, n_kv_heads=kv_heads, rms_eps=EPS, rope_theta=THETA,
                 max_position=PAGE * int(tables.shape[1]), num_blocks=num_blocks, max_batch_tokens=max(64, sum(new)),
                 max_seqs=max(4, len(ctx)), dtype=dtype)
    g = _gen(seed)
    pools = [[_pool(kv, layer, w).normal_(generator=g) for w in "kv"] for layer in range(case["layers"])]
    return kv, pools, (ctx, new, tables), g


# ---- step ----------------------------------------------------------------------------------------------


def _step_inputs(case: dict, g, T: int):
    dt = torch.float16 if case["dtype"] == "f16" else torch.float32
    width = (case["heads"] + 2 * case["kv_heads"]) * D
    return [(_normal(g, T, width, dtype=dt), _norm_weight(g, D), _norm_weight(g, D)) for _ in range(case["layers"])]


def _prepare_step(case: dict, seed: int):
    dt = torch.float16 if case["dtype"] == "f16" else torch.float32
    kv, pools, (ctx, new, tables), g = _kv(case, seed, case["heads"], case["kv_heads"], dt)
    T = sum(new)
    inputs = _step_inputs(case, g, T)
    outs = [torch.empty(T, case["heads"], D, dtype=dt, device="cuda") for _ in inputs]
    return dict(kv=kv, pools=pools, batch=_batch(ctx, new, tables), inputs=inputs, outs=outs)


def _run_step(s):
    kv = s["kv"]
    kv.plan(s["batch"])
    for layer, ((qkv, qn, kn), out) in enumerate(zip(s["inputs"], s["outs"])):
        kv.layer(layer, qkv, out, qn, kn)
    return {"out": s["outs"], "pools": s["pools"]}


# ---- block ---------------------------------------------------------------------------------------------


def _block_inputs(case: dict, g, T: int):
    hidden = SHAPES[case["model"]][0]
    h = torch.randn(T, hidden, generator=g, device="cuda")
    per = [(_norm_weight(g, hidden), _normal(g, 32 * D, hidden, scale=0.02), _normal(g, hidden, 16 * D, scale=0.02),
            _norm_weight(g, D), _norm_weight(g, D)) for _ in range(case["layers"])]
    return h, per


def _prepare_block(case: dict, seed: int):
    kv, pools, (ctx, new, tables), g = _kv(case, seed, 16, 8)
    T = sum(new)
    h, per = _block_inputs(case, g, T)
    hidden = h.shape[1]
    f16 = dict(dtype=torch.float16, device="cuda")
    return dict(kv=kv, pools=pools, batch=_batch(ctx, new, tables), h=h, per=per, xn=torch.empty(T, hidden, **f16),
                qkv=torch.empty(T, 32 * D, **f16), att=torch.empty(T, 16, D, **f16))


def _run_block(s):
    """The residual runs on from pass to pass, as it does from layer to layer."""
    kv = s["kv"]
    kv.plan(s["batch"])
    for layer, (norm, w_qkv, w_o, qn, kn) in enumerate(s["per"]):
        kv.attention_block(layer, s["h"], norm, w_qkv, w_o, xn=s["xn"], qkv=s["qkv"], att=s["att"], q_norm=qn, k_norm=kn)
    return {"h": s["h"], "pools": s["pools"]}


# ---- mlp -----------------------------------------------------------------------------------------------


def _mlp_inputs(case: dict, seed: int):
    hidden, inter = SHAPES[case["model"]]
    g = _gen(seed)
    return (torch.randn(case["tokens"], hidden, generator=g, device="cuda"), _norm_weight(g, hidden),
            _normal(g, 2 * inter, hidden, scale=0.02), _normal(g, hidden, inter, scale=0.02))


def _prepare_mlp(case: dict, seed: int):
    h, norm, gate_up, down = _mlp_inputs(case, seed)
    T, hidden, inter = h.shape[0], h.shape[1], down.shape[1]
    need = max(int(_lib.lib().ember_hip_gemv_workspace_bytes(64, *w.shape)) for w in (gate_up, down))
    return dict(h=h, norm=norm, gate_up=gate_up, down=down,
                packed=[K.gemv_pack(w) if case["packed"] else None for w in (gate_up, down)],
                ws=torch.zeros(need, dtype=torch.uint8, device="cuda") if need else None,
                xn=torch.empty(T, hidden, dtype=torch.float16, device="cuda"),
                act=torch.empty(T, inter, dtype=torch.float16, device="cuda"))


def _run_mlp(s):
    K.rmsnorm_rows(s["h"], s["norm"], s["xn"], EPS)
    K.gemv(s["xn"], s["gate_up"], s["act"], _lib.EPILOGUE_SILU_MUL, workspace=s["ws"], packed=s["packed"][0])
    K.gemv(s["act"], s["down"], s["h"], _lib.EPILOGUE_ADD_F32, workspace=s["ws"], packed=s["packed"][1])
    return {"act": s["act"], "h": s["h"]}


# ---- sample --------------------------------------------------------------------------------------------


def _logits(case: dict, seed: int):
    """Rows as a language model gives them: a broad floor, a few dozen likely tokens well above it."""
    R, V = case["rows"], case["vocab"]
    g = _gen(seed)
    x = 2.0 * torch.randn(R, V, generator=g, device="cuda")
    likely = torch.randint(V, (R, 64), generator=g, device="cuda")
    x.scatter_add_(1, likely, 8.0 + 6.0 * torch.rand(R, 64, generator=g, device="cuda"))
    return x, likely[:, 0].to(torch.int32).contiguous()


def _prepare_sample(case: dict, seed: int):
    x, drafts = _logits(case, seed)
    R, V = x.shape
    p = (_lib.SampleParams * R)()
    for i in range(R):
        p[i].temperature, p[i].top_p, p[i].top_k, p[i].min_p = case["temperature"], case["top_p"], case["top_k"], case["min_p"]
        p[i].seed, p[i].counter = seed * 1000 + i, 17 * i
    params = torch.frombuffer(bytearray(p), dtype=torch.uint8).cuda()
    rows = torch.arange(R, dtype=torch.int32, device="cuda")
    tokens = torch.empty(R, dtype=torch.int32, device="cuda")
    probs = torch.empty(R, device="cuda")
    a, b = _lib.SampleArgs(), _lib.ProbArgs()
    a.logits, a.R, a.vocab, a.params, a.out = x.data_ptr(), R, V, params.data_ptr(), tokens.data_ptr()
    b.logits, b.vocab, b.params, b.rows, b.tokens = x.data_ptr(), V, params.data_ptr(), rows.data_ptr(), drafts.data_ptr()
    b.n, b.out, b.R = R, probs.data_ptr(), R
    return dict(a=a, b=b, tokens=tokens, probs=probs, keep=(x, params, rows, drafts))


def _run_sample(s):
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.lib().ember_hip_sample(ctypes.byref(s["a"]), stream), "sample")
    _lib.check(_lib.lib().ember_hip_token_probs(ctypes.byref(s["b"]), stream), "token_probs")
    return {"tokens": s["tokens"], "probs": s["probs"]}


# ---- backend -------------------------------------------------------------------------------------------

LAYERS = 28
HID, INTER = SHAPES["0.6B"]
GREEDY = SamplingParams(temperature=0.0)


def _weights():
    """(name, f16 tensor on the GPU) of the model directory, in order: N(0, 0.02), norms about one."""
    g = _gen(7)
    yield "model.embed_tokens.weight", _normal(g, VOCAB, HID, scale=0.02)
    yield "model.norm.weight", _norm_weight(g, HID).half()
    for layer in range(LAYERS):
        p = f"model.layers.{layer}."
        for name, rows, cols in (("self_attn.q_proj", 16 * D, HID), ("self_attn.k_proj", 8 * D, HID),
                                 ("self_attn.v_proj", 8 * D, HID), ("self_attn.o_proj", HID, 16 * D),
                                 ("mlp.gate_proj", INTER, HID), ("mlp.up_proj", INTER, HID), ("mlp.down_proj", HID, INTER)):
            yield p + name + ".weight", _normal(g, rows, cols, scale=0.02)
        for name, n in (("input_layernorm", HID), ("post_attention_layernorm", HID), ("self_attn.q_norm", D),
                        ("self_attn.k_norm", D)):
            yield p + name + ".weight", _norm_weight(g, n).half()


@functools.lru_cache(maxsize=1)
def _model_dir() -> str:
    """The model directory, written once: what a user has downloaded before the program starts."""
    path = tempfile.mkdtemp(prefix="ember_cases_")
    tensors = [(n, t.cpu().numpy()) for n, t in _weights()]
    header, at = {}, 0
    for n, t in tensors:
        header[n] = {"dtype": "F16", "shape": list(t.shape), "data_offsets": [at, at + t.nbytes]}
        at += t.nbytes
    head = json.dumps(header).encode()
    with open(os.path.join(path, "model.safetensors"), "wb") as f:
        f.write(len(head).to_bytes(8, "little") + head)
        for _, t in tensors:
            t.tofile(f)
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(dict(model_type="qwen3", vocab_size=VOCAB, hidden_size=HID, intermediate_size=INTER,
                       num_hidden_layers=LAYERS, num_attention_heads=16, num_key_value_heads=8, head_dim=D,
                       rms_norm_eps=EPS, rope_theta=THETA, max_position_embeddings=2048, tie_word_embeddings=True,
                       eos_token_id=2), f)
    return path


def _prompts(case: dict, seed: int) -> np.ndarray:
    """Token ids [seqs, tokens (+ 1 for the decode step)]."""
    n = case["tokens"] + (case["phase"] == "decode")
    return np.random.default_rng(seed).integers(3, VOCAB, (case["seqs"], n)).astype(np.int32)


def _prepare_backend(case: dict, seed: int):
    ids, S, n = _prompts(case, seed), case["seqs"], case["tokens"]
    width = (n + 1 + PAGE - 1) // PAGE
    be = create_backend(_model_dir(), BackendOptions(max_batch_tokens=max(64, S * n), max_seqs=max(8, S),
                                                     kv_cache_tokens=max(64, S * width * PAGE)))
    tables = np.random.default_rng(seed + 1).permutation(S * width).astype(np.int32).reshape(S, width)

    def batch(first, count):
        b = _batch([first + count] * S, [count] * S, tables)
        b.tokens = np.ascontiguousarray(ids[:, first:first + count]).reshape(-1)
        b.logit_rows = [count * (i + 1) - 1 for i in range(S)]
        return b

    step = batch(0, n)
    if case["phase"] == "decode":  # the prompts are in the cache
        be.forward(step)
        be.sample([SampleRequest(GREEDY)] * S)
        step = batch(n, 1)
    return dict(be=be, step=step, S=S)


def _run_backend(s):
    be, S = s["be"], s["S"]
    be.forward(s["step"])
    tokens = be.sample([SampleRequest(GREEDY)] * S)
    return {"logits": [be.logits(i) for i in range(S)], "tokens": tokens}


# ---- the interface -------------------------------------------------------------------------------------

PREPARE = dict(step=_prepare_step, block=_prepare_block, mlp=_prepare_mlp, sample=_prepare_sample, backend=_prepare_backend)
RUN = dict(step=_run_step, block=_run_block, mlp=_run_mlp, sample=_run_sample, backend=_run_backend)


def prepare(case: dict, seed: int):
    return {"kind": case["kind"], **PREPARE[case["kind"]](case, seed)}


def run(state):
    return RUN[state["kind"]](state)


def _attention_work(ctx, new, heads, kv_heads, es, prefix=0):
    """(bytes, flops) of one layer's append + attention; a shared prefix is read once."""
    tokens, T = prefix + sum(c - prefix for c in ctx), sum(new)
    cached = tokens - T
    pairs = sum(n * c - n * (n - 1) // 2 for c, n in zip(ctx, new))  # (query, key) pairs under the causal mask
    kv = 2 * kv_heads * D * es
    per_token = (heads + 2 * kv_heads) * D * es + kv + heads * D * es  # qkv in, K/V out, attention out
    return cached * kv + T * per_token, 4 * D * heads * pairs


def _linear_work(M, N, Kd, out_bytes):
    return 2 * N * Kd + 2 * M * Kd + out_bytes, 2 * M * N * Kd


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "step":
        es = 2 if case["dtype"] == "f16" else 4
        b, f = _attention_work(_contexts(case), _new_tokens(case), case["heads"], case["kv_heads"], es, case["prefix"])
        return {"bytes": b * case["layers"], "flops": f * case["layers"]}
    if kind == "sample":
        return {"bytes": 4 * case["rows"] * case["vocab"], "flops": 2 * case["rows"] * case["vocab"]}
    if kind == "mlp":
        hidden, inter = SHAPES[case["model"]]
        T = case["tokens"]
        parts = [(8 * T * hidden, 4 * T * hidden), _linear_work(T, 2 * inter, hidden, 0), _linear_work(T, hidden, inter, 2 * T * inter)]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    if kind == "block":
        hidden = SHAPES[case["model"]][0]
        ctx, new = _contexts(case), _new_tokens(case)
        T = sum(new)
        parts = [_attention_work(ctx, new, 16, 8, 2), _linear_work(T, 32 * D, hidden, 8 * T * hidden),
                 _linear_work(T, hidden, 16 * D, 0)]
        return {"bytes": case["layers"] * sum(p[0] for p in parts), "flops": case["layers"] * sum(p[1] for p in parts)}
    S, n = case["seqs"], case["tokens"]
    new = n if case["phase"] == "prompt" else 1
    ctx = n if case["phase"] == "prompt" else n + 1
    per = 4 * HID * 1024 + HID * 2048 + 3 * HID * INTER  # weights of one layer
    b, f = _attention_work([ctx] * S, [new] * S, 16, 8, 2)
    T = S * new
    return {"bytes": LAYERS * (2 * per + b) + 2 * VOCAB * HID + 4 * S * VOCAB,
            "flops": LAYERS * (2 * T * per + f) + 2 * S * VOCAB * HID}


def tolerance(case: dict):
    """About four times what the outputs are seen to differ from exact() by: f16 roundings of the attention output,
    the MLP activation and a model's every layer; the block's residual adds small f16 terms to an f32 sum."""
    kind = case["kind"]
    if kind == "step":
        return {"rel": 2e-5, "max": 1e-3} if case["dtype"] == "f32" else {"rel": 1.5e-3, "max": 0.02}
    if kind == "block":
        return {"rel": 2e-4, "max": 0.02}
    if kind == "mlp":
        return {"rel": 1.5e-3, "max": 0.02}
    if kind == "sample":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}
    return {"rel": 4e-3, "max": 0.05, "differ": 0.01}


# ---- the same in 64 bits, by plain torch -------------------------------------------------------------


def _rms(x, w, eps=EPS):
    return w.double() * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _rope(x, pos):
    """Rotate-half RoPE of x [T, heads, 128]; the angle is an f32 position times an f32 frequency."""
    i = np.arange(D // 2, dtype=np.float32)
    freq = (np.float32(1.0) / np.power(np.float32(THETA), (2 * i) / np.float32(D), dtype=np.float32)).astype(np.float32)
    ang = (pos.float()[:, None] * torch.from_numpy(freq).to(pos.device)).double()[:, None, :]
    c, s = ang.cos(), ang.sin()
    lo, hi = x[..., : D // 2], x[..., D // 2:]
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _exact_attention(qkv, qn, kn, kp, vp, ctx, new, tables, heads, kv_heads, out_pools=True):
    """One layer's append + attention in 64 bits. qkv [T, ...] f64; kp / vp: the pools as given. Returns (out, K pool, V pool)."""
    T, G = qkv.shape[0], heads // kv_heads
    pos = torch.cat([torch.arange(c - n, c) for c, n in zip(ctx, new)]).cuda()
    q, k, v = qkv[:, : heads * D], qkv[:, heads * D: (heads + kv_heads) * D], qkv[:, (heads + kv_heads) * D:]
    q = _rope(_rms(q.reshape(T, heads, D), qn), pos)
    k = _rope(_rms(k.reshape(T, kv_heads, D), kn), pos)
    v = v.reshape(T, kv_heads, D)
    out = torch.empty(T, heads, D, dtype=torch.float64, device="cuda")
    at, blocks = 0, torch.from_numpy(tables).cuda().long()
    new_block, new_slot = [], []
    for s, (c, n) in enumerate(zip(ctx, new)):
        pages = blocks[s, : (c + PAGE - 1) // PAGE]
        kk = kp[pages].double().transpose(1, 2).reshape(-1, kv_heads, D)[:c].clone()
        vv = vp[pages].double().transpose(1, 2).reshape(-1, kv_heads, D)[:c].clone()
        kk[c - n:], vv[c - n:] = k[at:at + n], v[at:at + n]
        qs = q[at:at + n].reshape(n, kv_heads, G, D).permute(1, 2, 0, 3).reshape(kv_heads, G * n, D)
        mask = torch.arange(c, device="cuda")[None, :] > torch.arange(c - n, c, device="cuda")[:, None]  # [n, c]
        for h in range(kv_heads):  # one kv head at a time: bounded memory
            sc = (qs[h] @ kk[:, h].T.contiguous()) / math.sqrt(D)
            sc.reshape(G, n, c).masked_fill_(mask, -math.inf)
            o = torch.softmax(sc, -1) @ vv[:, h].contiguous()
            out[at:at + n, h * G:(h + 1) * G] = o.reshape(G, n, D).transpose(0, 1)
        p = torch.arange(c - n, c, device="cuda")
        new_block.append(blocks[s][p // PAGE])
        new_slot.append(p % PAGE)
        at += n
    if not out_pools:
        return out, k, v
    b, sl = torch.cat(new_block), torch.cat(new_slot)
    kd, vd = kp.double(), vp.double()
    kd[b, :, sl], vd[b, :, sl] = k, v
    return out, kd, vd


def _pools(case: dict, g, num_blocks: int, kv_heads: int, dt):
    """The pages prepare() fills, drawn alike."""
    make = lambda: torch.empty(num_blocks + 1, kv_heads, PAGE, D, dtype=dt, device="cuda").normal_(generator=g)  # noqa: E731
    return [[make(), make()] for _ in range(case["layers"])]


def _exact_step(case: dict, seed: int):
    dt = torch.float16 if case["dtype"] == "f16" else torch.float32
    ctx, new, tables, num_blocks = _layout(case, seed)
    g = _gen(seed)
    pools = _pools(case, g, num_blocks, case["kv_heads"], dt)
    outs, after = [], []
    for (qkv, qn, kn), (kp, vp) in zip(_step_inputs(case, g, sum(new)), pools):
        o, kd, vd = _exact_attention(qkv.double(), qn, kn, kp, vp, ctx, new, tables, case["heads"], case["kv_heads"])
        outs.append(o)
        after.append([kd, vd])
    return {"out": outs, "pools": after}


def _exact_block(case: dict, seed: int):
    ctx, new, tables, num_blocks = _layout(case, seed)
    g = _gen(seed)
    pools = _pools(case, g, num_blocks, 8, torch.float16)
    h, per = _block_inputs(case, g, sum(new))
    h, after = h.double(), []
    for (norm, w_qkv, w_o, qn, kn), (kp, vp) in zip(per, pools):
        qkv = _rms(h, norm) @ w_qkv.double().T
        o, kd, vd = _exact_attention(qkv, qn, kn, kp, vp, ctx, new, tables, 16, 8)
        h = h + o.reshape(len(h), -1) @ w_o.double().T
        after.append([kd, vd])
    return {"h": h, "pools": after}


def _silu_mul(x, gate_up):
    y = x @ gate_up.double().T
    return torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2]


def _exact_mlp(case: dict, seed: int):
    h, norm, gate_up, down = _mlp_inputs(case, seed)
    h = h.double()
    act = _silu_mul(_rms(h, norm), gate_up)
    return {"act": act, "h": h + act @ down.double().T}


def _exact_sample(case: dict, seed: int):
    """The drafted tokens' probabilities: temperature, top-k, top-p over its mass, min-p; greedy rows one or zero."""
    x, drafts = _logits(case, seed)
    drafts = drafts.long()[:, None]
    if case["temperature"] <= 1e-5:
        return {"tokens": None, "probs": (x.argmax(-1, keepdim=True) == drafts)[:, 0].double()}
    # the scaled logit is an f32 quotient; the order is by it, then by id
    v, order = torch.sort((x / case["temperature"]).double(), dim=-1, descending=True, stable=True)
    keep = torch.ones_like(v, dtype=torch.bool)
    if 0 < case["top_k"] < case["vocab"]:
        keep[:, case["top_k"]:] = False
    w = torch.exp(v - v[:, :1]) * keep
    if case["top_p"] < 1.0:
        before = w.cumsum(-1) - w
        keep &= before < case["top_p"] * w.sum(-1, keepdim=True)
    keep &= torch.exp(v - v[:, :1]) >= case["min_p"]
    w = w * keep
    p = torch.zeros_like(v).scatter_(1, order, w / w.sum(-1, keepdim=True))
    return {"tokens": None, "probs": p.gather(1, drafts)[:, 0]}


def _exact_backend(case: dict, seed: int):
    ids, S = _prompts(case, seed), case["seqs"]
    n = ids.shape[1]
    W = dict(_weights())
    logits = []
    for s in range(S):
        h = W["model.embed_tokens.weight"][torch.from_numpy(ids[s]).cuda().long()].double()
        tables = np.arange((n + PAGE - 1) // PAGE, dtype=np.int32)[None, :]
        empty = torch.zeros(tables.size, 8, PAGE, D, dtype=torch.float16, device="cuda")
        for layer in range(LAYERS):
            w = lambda k: W[f"model.layers.{layer}.{k}.weight"]  # noqa: E731
            x = _rms(h, w("input_layernorm"))
            qkv = torch.cat([x @ w(f"self_attn.{t}_proj").double().T for t in "qkv"], -1)
            o, _, _ = _exact_attention(qkv, w("self_attn.q_norm"), w("self_attn.k_norm"), empty, empty, [n], [n], tables, 16, 8, False)
            h = h + o.reshape(n, -1) @ w("self_attn.o_proj").double().T
            x = _rms(h, w("post_attention_layernorm"))
            act = torch.nn.functional.silu(x @ w("mlp.gate_proj").double().T) * (x @ w("mlp.up_proj").double().T)
            h = h + act @ w("mlp.down_proj").double().T
        x = _rms(h[-1:], W["model.norm.weight"])
        logits.append((x @ W["model.embed_tokens.weight"].double().T)[0])
    return {"logits": logits, "tokens": None}


EXACT = dict(step=_exact_step, block=_exact_block, mlp=_exact_mlp, sample=_exact_sample, backend=_exact_backend)


def exact(case: dict, seed: int):
    return EXACT[case["kind"]](case, seed)
