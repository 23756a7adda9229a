"""Measured cases of the hybrid-cache framework: what a serving loop on this library calls, per step and per layer.

Sizes are those of the two OPT shapes the repository carries (12 x 64 and 40 x 128 heads), the batches
``workloads`` and ``step_loop`` generate (lognormal lengths up to 2048 tokens, half of the sequences
hidden-cached, 16-token blocks), and what lies between them.  A case names its sizes; the lengths of its
sequences follow from them (quantiles of the lognormal, scaled to the stated total), the seed decides the order
of the sequences, where their blocks lie and every value.
"""

from __future__ import annotations

import math
import os
import statistics
import sys
from types import SimpleNamespace

import numpy as np
import torch

_PACKAGE = os.path.join(os.getcwd(), "apt-serve_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from aptserve_hip import metadata, ops, workloads  # noqa: E402
from aptserve_hip.backend import HybridOPTAttention  # noqa: E402
from aptserve_hip.graph_step import DecodeGraphRunner  # noqa: E402
from aptserve_hip.opt_model import HybridOPTModel, OPTConfig, random_weights  # noqa: E402

BS = workloads.BLOCK_SIZE
MAX_LEN = 2048
_MODELS = {"opt_125m": workloads.OPT_125M, "opt_13b": workloads.OPT_13B}
_DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "fp8": torch.float16}
_KV_SCALE = 0.04        # per-tensor scale of an fp8 K/V cache holding N(0, 1) rows


def listed():
    return [
        # Cache write of a small prompt step on the small model: eight short prompts, some hidden-cached.  A launch
        # and its checks: what the smallest calls of the library cost.
        dict(name="prompt_write_125m", op="prompt_write", model="opt_125m", dtype="f16", seqs=8, tokens=351, hidden=0.3),
        # The cache traffic of one layer of a full decode step (256 sequences, half hidden-cached): new rows stored,
        # every cached hidden row gathered for the re-projection.
        dict(name="decode_store_256", op="decode_store", model="opt_13b", dtype="f16", seqs=256, tokens=173500, hidden=0.5),
        # Decode attention of a large batch whose sequences lie half in the K/V cache, half in the re-projected workspace.
        dict(name="decode_attn_f16", op="decode_attn", model="opt_13b", dtype="f16", seqs=128, tokens=86500, hidden=0.5),
        # The same on an fp8 cache, which serves twice the tokens in the same memory.
        dict(name="decode_attn_fp8", op="decode_attn", model="opt_13b", dtype="fp8", seqs=128, tokens=86500, hidden=0.5),
        # Ragged-batch metadata of a full decode step from packed block tables: once per step, before any layer.
        dict(name="metadata_256", op="metadata", model="opt_13b", dtype="f16", seqs=256, tokens=173500, hidden=0.5,
             packed=True),
        # K/V re-projection of a layer's gathered hidden rows, the largest plain matrix product of the path.
        dict(name="reproject_16384", op="reproject", model="opt_13b", dtype="f16", rows=16384),
        # Causal attention of a large prompt step: four prompts of the longest length served.
        dict(name="prompt_attn_4x2048", op="prompt_attn", model="opt_13b", dtype="f16", seqs=4, tokens=8192, context=0),
        # Chunked prompts: the new tokens of each sequence attend to its cached prefix through the block table.
        dict(name="prompt_attn_prefix_bf16", op="prompt_attn", model="opt_13b", dtype="bf16", seqs=6, tokens=2048,
             context=4200),
        # Self-attention of a decoder layer in the reference's data flow (hidden rows re-projected every step),
        # a medium batch in bf16.
        dict(name="layer_reproject_24", op="layer", model="opt_13b", dtype="bf16", seqs=24, tokens=16000, hidden=0.5,
             absorbed=False),
        # Self-attention of a decoder layer on the cached hidden rows themselves, a full batch.
        dict(name="layer_absorbed_256", op="layer", model="opt_13b", dtype="f16", seqs=256, tokens=173500, hidden=0.5,
             absorbed=True),
        # A whole decode step of the 40-layer decoder at the batch a steady stream of requests settles at,
        # metadata included, replayed from its HIP graph.
        dict(name="model_decode_5", op="model_decode", model="opt_13b", dtype="f16", seqs=5, tokens=1180, hidden=0.6,
             layers=40),
        # A whole prompt step of the 40-layer decoder (one long and one short prompt), metadata included.
        dict(name="model_prompt_361", op="model_prompt", model="opt_13b", dtype="f16", seqs=2, tokens=361, hidden=0.5,
             layers=40),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["prompt_write", "decode_store", "decode_attn", "metadata", "reproject", "prompt_attn", "layer",
                     "model_decode", "model_prompt"])
    dtype = rng.choice(["f16", "bf16"])
    model = rng.choice(["opt_13b", "opt_13b", "opt_125m"])
    hidden = round(rng.uniform(0.0, 1.0), 3)
    if op == "prompt_write":
        tokens = _log(rng, 8, 16384)
        return dict(op=op, model=model, dtype=dtype, seqs=max(-(-tokens // MAX_LEN), min(tokens, _log(rng, 1, 32))),
                    tokens=tokens, hidden=hidden)
    if op == "decode_store":
        seqs = _log(rng, 1, 256)
        return dict(op=op, model=model, dtype=dtype, seqs=seqs, tokens=_decode_tokens(rng, seqs), hidden=hidden)
    if op == "decode_attn":
        seqs = _log(rng, 1, 128)
        return dict(op=op, model=model, dtype=rng.choice(["f16", "bf16", "fp8"]), seqs=seqs,
                    tokens=_decode_tokens(rng, seqs), hidden=hidden)
    if op == "metadata":
        seqs = _log(rng, 1, 256)
        return dict(op=op, model="opt_13b", dtype=dtype, seqs=seqs, tokens=_decode_tokens(rng, seqs), hidden=hidden,
                    packed=rng.random() < 0.7)
    if op == "reproject":
        return dict(op=op, model=model, dtype=dtype, rows=_log(rng, 16, 16384))
    if op == "prompt_attn":
        tokens = _log(rng, 16, 8192)
        seqs = max(-(-tokens // MAX_LEN), min(tokens, _log(rng, 1, 16)))
        context = rng.choice([0, 0, _log(rng, seqs, max(seqs, min(8192, seqs * MAX_LEN // 2)))])
        return dict(op=op, model=model, dtype=dtype, seqs=seqs, tokens=tokens, context=context)
    if op == "layer":
        absorbed = rng.random() < 0.5
        seqs = _log(rng, 1, 256 if absorbed else 64)
        return dict(op=op, model="opt_13b", dtype=dtype, seqs=seqs, tokens=_decode_tokens(rng, seqs), hidden=hidden,
                    absorbed=absorbed)
    if op == "model_decode":
        seqs = _log(rng, 1, 32)
        return dict(op=op, model=model, dtype=dtype, seqs=seqs, tokens=_decode_tokens(rng, seqs), hidden=hidden,
                    layers=rng.randint(4, 24 if model == "opt_13b" else 12))
    tokens = _log(rng, 16, 4096)
    return dict(op=op, model=model, dtype=dtype, seqs=max(-(-tokens // MAX_LEN), min(tokens, _log(rng, 1, 8))),
                tokens=tokens, hidden=hidden, layers=max(1, min(40 if model == "opt_13b" else 12, 361 * 40 // tokens)))


def _decode_tokens(rng, seqs):
    """Total cached length of a decode batch: a mean per sequence from 16 tokens to 700 (what lognormal(6.2, 0.8) has)."""
    return max(seqs, _log(rng, 16 * seqs, 700 * seqs))


# ------------------------------------------------------------------------------- the batch a case stands for

def _lengths(n, total, longest=MAX_LEN):
    """``n`` lengths of ``total`` tokens in all, at the quantiles of a lognormal of sigma 0.8, none above ``longest``."""
    z = statistics.NormalDist()
    w = [math.exp(0.8 * z.inv_cdf((i + 0.5) / n)) for i in range(n)]
    lo, hi = 0.0, 1e9
    for _ in range(200):                    # the scale at which the clipped lengths add up to the total
        mid = (lo + hi) / 2
        if sum(min(longest, max(1.0, mid * x)) for x in w) < total:
            lo = mid
        else:
            hi = mid
    lens = [int(min(longest, max(1.0, hi * x))) for x in w]
    k = 0
    while sum(lens) < total and k < 4 * n:  # what rounding down left over, one token each, longest first
        i = n - 1 - k % n
        if lens[i] < longest:
            lens[i] += 1
        k += 1
    return lens


def _flags(n, fraction):
    """``round(fraction * n)`` hidden-cached sequences, spread evenly over the sorted lengths."""
    return [int((i + 1) * fraction + 0.5) > int(i * fraction + 0.5) for i in range(n)]


def _sizes(case):
    m = _MODELS[case["model"]]
    return m["num_heads"], m["head_size"], m["hidden_size"]


def _batch(case, seed, is_prompt):
    lens, flags = _lengths(case["seqs"], case["tokens"]), _flags(case["seqs"], case["hidden"])
    rng = np.random.default_rng(seed)
    order = rng.permutation(len(lens))
    lens, flags = [lens[i] for i in order], [flags[i] for i in order]
    need = sum(-(-n // BS) for n in lens)
    return workloads.allocate_blocks(rng, lens, flags, max(64, need + need // 4), BS, is_prompt)


def _split(case):
    """(tokens of hidden-cached sequences, number of them, all tokens, number of sequences)"""
    lens, flags = _lengths(case["seqs"], case["tokens"]), _flags(case["seqs"], case["hidden"])
    return sum(n for n, f in zip(lens, flags) if f), sum(flags), sum(lens), len(lens)


# ------------------------------------------------------------------------------- inputs

def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _randn(g, *shape, dtype=torch.float16, std=1.0):
    x = torch.randn(*shape, generator=g, device=g.device, dtype=dtype)
    return x if std == 1.0 else x.mul_(std)


def _codes(g, *shape):
    """fp8-e4m3 codes of N(0, 1) rows at the scale the cache is read with."""
    x = torch.empty(*shape, dtype=torch.uint8, device=g.device)
    for i in range(0, shape[1], 4096):
        r = torch.randn(shape[0], min(4096, shape[1] - i), *shape[2:], generator=g, device=g.device)
        x[:, i:i + 4096] = torch.clamp(r / _KV_SCALE, -448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    return x


def prepare(case, seed):
    op = case["op"]
    dev = _device()
    g = torch.Generator(device=dev).manual_seed(seed)
    H, D, Hd = _sizes(case)
    dt = _DTYPES[case["dtype"]]
    s = SimpleNamespace(op=op, heads=H, scale=D ** -0.5)
    if op == "prompt_write":
        b = _batch(case, seed, True)
        s.md = metadata.build_from_batch(b, dev)
        T = s.md.num_prefill_tokens
        s.k, s.v = _randn(g, T, 3 * Hd, dtype=dt).chunk(3, -1)[1:]      # as they leave the fused projection
        s.hidden = _randn(g, T, Hd, dtype=dt)
        s.cache = torch.zeros(2, b.num_blocks, BS, H, D, dtype=dt, device=dev)
    elif op == "decode_store":
        b = _batch(case, seed, False)
        s.md = metadata.build_from_batch(b, dev)
        B = case["seqs"]
        s.k, s.v = _randn(g, B, 3 * Hd, dtype=dt).chunk(3, -1)[1:]
        s.hidden = _randn(g, B, Hd, dtype=dt)
        s.cache = _randn(g, 2, b.num_blocks, BS, H, D, dtype=dt)
        s.holder = torch.empty(s.md.num_tot_tokens, Hd, dtype=dt, device=dev)
    elif op == "decode_attn":
        b = _batch(case, seed, False)
        s.md = metadata.build_from_batch(b, dev)
        N = b.num_blocks
        s.q = _randn(g, case["seqs"], H, D, dtype=dt)
        make = _codes if case["dtype"] == "fp8" else (lambda g, *sh: _randn(g, *sh, dtype=dt))
        s.kv_scale = _KV_SCALE if case["dtype"] == "fp8" else None
        s.cache = make(g, 2, N, BS, H, D)
        s.workspace = make(g, 2, 2 * N, BS, H, D) if s.md.block_types is not None else None
    elif op == "metadata":
        s.batch, s.packed, s.dev = _batch(case, seed, False), case["packed"], dev
        s.batch.packed_tables()             # a block manager keeps its tables in this form
    elif op == "reproject":
        s.w, s.b = _randn(g, 2 * Hd, Hd, dtype=dt, std=0.02), _randn(g, 2 * Hd, dtype=dt, std=0.02)
        s.x = _randn(g, case["rows"], Hd, dtype=dt)
    elif op == "prompt_attn":
        rng = np.random.default_rng(seed)
        lens = _lengths(case["seqs"], case["tokens"])
        order = rng.permutation(len(lens))
        lens = [lens[i] for i in order]
        T, s.max_q = sum(lens), max(lens)
        s.cu_q = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32).to(dev)
        s.context = case["context"]
        if not s.context:
            s.q, s.k, s.v = (x.view(T, H, D) for x in _randn(g, T, 3 * Hd, dtype=dt).chunk(3, -1))
        else:
            ctx = _lengths(case["seqs"], case["context"], longest=MAX_LEN * 4)
            tot = [n + c for n, c in zip(lens, [ctx[i] for i in rng.permutation(len(ctx))])]
            need = sum(-(-n // BS) for n in tot)
            b = workloads.allocate_blocks(rng, tot, [False] * len(tot), max(64, need + need // 4), BS, True)
            s.table = torch.from_numpy(b.packed_tables()[0]).to(dev)
            s.cu_k = torch.tensor(np.concatenate([[0], np.cumsum(tot)]), dtype=torch.int32).to(dev)
            s.max_k = max(tot)
            s.q = _randn(g, T, H, D, dtype=dt)
            s.cache = _randn(g, 2, b.num_blocks, BS, H, D, dtype=dt)
    elif op == "layer":
        b = _batch(case, seed, False)
        s.md = metadata.build_from_batch(b, dev)
        w, bias = _randn(g, 3 * Hd, Hd, dtype=dt, std=0.02), _randn(g, 3 * Hd, dtype=dt, std=0.02)
        ow, ob = _randn(g, Hd, Hd, dtype=dt, std=0.02), _randn(g, Hd, dtype=dt, std=0.02)
        s.layer = HybridOPTAttention(Hd, H, w, bias, ow, ob, absorbed=case["absorbed"])
        s.hidden = _randn(g, case["seqs"], Hd, dtype=dt)
        s.cache = _randn(g, 2, b.num_blocks, BS, H, D, dtype=dt)
        s.shared = torch.zeros(2, 2 * b.num_blocks, BS, H, D, dtype=dt, device=dev)
    else:
        b = s.batch = _batch(case, seed, op == "model_prompt")
        L = case["layers"]
        cfg = OPTConfig.opt_13b() if case["model"] == "opt_13b" else OPTConfig.opt_125m()
        s.model = HybridOPTModel(cfg, random_weights(cfg, seed, dev, dtype=dt, layers=L), num_layers=L, absorbed=True)
        s.caches = [_randn(g, 2, b.num_blocks, BS, H, D, dtype=dt) for _ in range(L)]
        s.shared = torch.zeros(2, 2 * b.num_blocks, BS, H, D, dtype=dt, device=dev)
        n = len(b.seq_lens) if op == "model_decode" else sum(b.seq_lens)
        s.ids = torch.from_numpy(np.random.default_rng(seed + 1).integers(0, cfg.vocab_size, n)).pin_memory()
        s.dev = dev
        if op == "model_decode":            # the graph of this step's shape class, recorded on its first step
            s.runner = DecodeGraphRunner(s.model, s.caches, s.shared, BS, dev)
            s.runner.step(b.seq_lens, b.use_hidden, b.block_tables, b.block_tables_4_shared, s.ids.to(dev))
    return s


# ------------------------------------------------------------------------------- one pass

def run(s):
    op = s.op
    if op == "prompt_write":
        ops.mixed_reshape_and_cache(s.k, s.v, s.hidden, s.cache, s.md.slot_mapping, s.md.token_is_hidden)
        return s.cache
    if op == "decode_store":
        md = s.md
        ops.decode_step_cache_ops(s.holder, s.hidden, s.cache, md.holder_src, md.slot_mapping,
                                  md.hidden_cache_use_input, md.hidden_cache_store_tot, s.k, s.v,
                                  md.kv_cache_use_input, md.new_token_slot)
        return s.holder, s.cache
    if op == "decode_attn":
        md = s.md
        return ops.paged_hybrid_attention(s.q, s.cache, s.workspace, md.block_tables, md.block_types,
                                          md.seq_lens_tensor, s.scale, s.kv_scale, max_seq_len=md.max_decode_seq_len)
    if op == "metadata":
        md = metadata.build_from_batch(s.batch, s.dev, packed=s.packed)
        return {k: v for k, v in vars(md).items() if isinstance(v, torch.Tensor)}
    if op == "reproject":
        return ops.kv_reproject(s.x, s.w, s.b)
    if op == "prompt_attn":
        if s.context:
            return ops.flash_attn_varlen_func(s.q, s.cache[0], s.cache[1], cu_seqlens_q=s.cu_q, cu_seqlens_k=s.cu_k,
                                              max_seqlen_q=s.max_q, max_seqlen_k=s.max_k, softmax_scale=s.scale,
                                              block_table=s.table)
        return ops.flash_attn_varlen_func(s.q, s.k, s.v, cu_seqlens_q=s.cu_q, cu_seqlens_k=s.cu_q,
                                          max_seqlen_q=s.max_q, max_seqlen_k=s.max_q, softmax_scale=s.scale)
    if op == "layer":
        return s.layer(s.hidden, s.cache, s.shared, s.md), s.cache
    b = s.batch
    if op == "model_decode":
        hidden, _ = s.runner.step(b.seq_lens, b.use_hidden, b.block_tables, b.block_tables_4_shared,
                                  s.ids.to(s.dev, non_blocking=True))
        return hidden, s.caches
    ids = s.ids.to(s.dev, non_blocking=True)
    md = metadata.build_from_batch(b, s.dev)
    return s.model(ids, md.input_positions, s.caches, s.shared, md), s.caches


# ------------------------------------------------------------------------------- what a pass cannot do without

def work(case):
    op = case["op"]
    H, D, Hd = _sizes(case)
    if op == "reproject":
        T = case["rows"]
        return {"bytes": 2 * (T * Hd + 2 * Hd * Hd + 2 * Hd + 2 * T * Hd), "flops": 4 * T * Hd * Hd}
    if op == "prompt_attn":
        lens, ctx = _lengths(case["seqs"], case["tokens"]), case["context"]
        T = sum(lens)
        pairs = sum(n * (n + 1) // 2 for n in lens)
        if ctx:                             # each new token also meets its sequence's prefix; prefixes in any order
            pairs += T * ctx // case["seqs"]
        return {"bytes": 2 * Hd * (2 * T + 2 * (T + ctx)), "flops": 4 * Hd * pairs}
    h_tok, h_seq, tok, seq = _split(case)
    kv_tok, kv_seq = tok - h_tok, seq - h_seq
    row = 2 * Hd                            # bytes of a hidden row, or of one K or V row, in 16 bits
    if op == "prompt_write":
        return {"bytes": 2 * row * (h_tok + 2 * kv_tok) + 9 * tok, "flops": 0}
    if op == "decode_store":
        return {"bytes": 2 * row * (h_tok + kv_seq + h_seq + 2 * kv_seq) + 8 * (h_tok + 2 * seq), "flops": 0}
    if op == "decode_attn":
        e = 1 if case["dtype"] == "fp8" else 2
        return {"bytes": 2 * Hd * e * tok + 2 * row * seq, "flops": 4 * Hd * tok}
    if op == "metadata":
        blocks = sum(-(-n // BS) for n in _lengths(case["seqs"], case["tokens"]))
        return {"bytes": 4 * 2 * blocks + 5 * blocks + 8 * (7 * h_tok + 8 * seq), "flops": 0}
    # the cached rows once (a hidden row, or K and V rows), the new rows, activations in and out
    cached = row * (h_tok + 2 * kv_tok)
    if op == "layer":
        out = {"bytes": 2 * 4 * Hd * Hd + cached + 2 * row * seq, "flops": 8 * seq * Hd * Hd + 4 * Hd * tok}
        if not case["absorbed"]:            # every hidden row is projected to its K and V rows, as this flow is defined
            out["flops"] += 4 * h_tok * Hd * Hd
        return out
    L, layer = case["layers"], 12 * Hd * Hd
    if op == "model_decode":
        return {"bytes": L * (2 * layer + cached) + 2 * row * seq, "flops": L * (2 * seq * layer + 4 * Hd * tok)}
    pairs = sum(n * (n + 1) // 2 for n in _lengths(case["seqs"], case["tokens"]))
    return {"bytes": L * (2 * layer + cached) + 2 * row * tok, "flops": L * (2 * tok * layer + 4 * Hd * pairs)}


#: (rel, max) a correct implementation may differ by: about four times what was measured against the path in 64 bits
#: (attention f16 2.7e-4, 4.0e-3, bf16 2.2e-3, 3.2e-2; re-projection 2.1e-4, 4.9e-4 and 1.7e-3, 3.9e-3), and for whole
#: layers and models, whose activations are rounded at every operator, between two flows of the same sums in another
#: order (layer 6.7e-4, 6.2e-3 and 5.6e-3, 4.0e-2; 40 layers 2.6e-3, 1.5e-2 and 2.0e-2, 1.1e-1).
_TOLERANCE = {
    "decode_attn": {"f16": (8e-4, 4e-3), "bf16": (6.6e-3, 3e-2)},
    "reproject": {"f16": (8e-4, 2e-3), "bf16": (6.6e-3, 1.6e-2)},
    "prompt_attn": {"f16": (1.1e-3, 1.6e-2), "bf16": (8.8e-3, 1.3e-1)},
    "layer": {"f16": (2.7e-3, 2.5e-2), "bf16": (2.2e-2, 1.6e-1)},
    "model_decode": {"f16": (1e-2, 6e-2), "bf16": (3e-2, 4e-1)},
    "model_prompt": {"f16": (1e-2, 6e-2), "bf16": (3e-2, 4e-1)},
}


def tolerance(case):
    """Byte moves and index vectors are exact; an fp8 cache is read exactly and computed on in fp16."""
    if case["op"] not in _TOLERANCE:
        return "exact"
    rel, most = _TOLERANCE[case["op"]]["bf16" if case["dtype"] == "bf16" else "f16"]
    return {"rel": rel, "max": most}
