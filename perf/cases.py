"""Timed cases of the serving hot path, through the package's public entry points.

A case is a dict of plain values; its kind says which entry point it goes through:

  decode   one new token per sequence over the paged pools: paged_attention_decode,
           or with `fused` the whole step (RoPE, KV append and attention),
           rope_append_paged_decode
  prefill  ragged chunks of prompts over the paged pools: paged_attention_prefill
  append   RoPE and the KV append of a packed iteration: rope_kv_append
  norm     RMSNorm with the residual add before it: rms_norm
  greedy   first-maximum token of every logits row: greedy_argmax
  model    one packed iteration of the whole model: LlamaModel.forward_packed

`prepare` builds what a serving program holds before the call, `run` is one call,
`exact` the same result in 64-bit torch. Sequence lengths follow from the case alone
(its `lengths` seed); values, block tables and weights from the seed given to `prepare`.
"""

from __future__ import annotations

import math
import random

import torch

from tokserve_amd.batching.metadata import PackedBatchBuilder, SequenceWork
from tokserve_amd.engine.config import tinyllama_1_1b
from tokserve_amd.engine.model import LlamaModel
from tokserve_amd.engine.paged.storage import PagedKVStorage
from tokserve_amd.kernels import ops

DEVICE = "cuda"
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
FP8 = torch.float8_e4m3fn
POOL_SCALES = (0.5, 0.25)  # k_scale, v_scale of fp8 pools with one scale per pool


def listed() -> list[dict]:
    return [
        # The smallest step: an fp32 layer of a small model serving a handful of requests.
        # Launches and latency count, not bytes.
        dict(name="decode_fp32_small", kind="decode", fused=True, dtype="float32", pool="same",
             seqs=8, min_keys=17, max_keys=513, log_keys=False, heads=8, kv_heads=2,
             head_dim=64, block_size=16, lengths=1),
        # One layer of a decode iteration at serving load, as the engine's decode calls it
        # (128 running requests of the 1.1B shape).
        dict(name="decode_serving_bf16", kind="decode", fused=True, dtype="bfloat16", pool="same",
             seqs=128, min_keys=65, max_keys=1152, log_keys=False, heads=32, kv_heads=4,
             head_dim=64, block_size=16, lengths=2),
        # Decode over long and short contexts of a full batch at the Llama-3-8B layer shape:
        # the headline of bench.py.
        dict(name="decode_long_bf16", kind="decode", fused=False, dtype="bfloat16", pool="same",
             seqs=256, min_keys=128, max_keys=8192, log_keys=True, heads=32, kv_heads=8,
             head_dim=128, block_size=16, lengths=0),
        # The same layer at an odd, middling batch over fp8 pools with a scale per row.
        dict(name="decode_fp8_rows", kind="decode", fused=False, dtype="bfloat16",
             pool="fp8_rows", seqs=33, min_keys=128, max_keys=8192, log_keys=True, heads=32,
             kv_heads=8, head_dim=128, block_size=16, lengths=4),
        # The block size is the pool owner's choice: 32 tokens to a block, fp16.
        dict(name="decode_block32_fp16", kind="decode", fused=False, dtype="float16", pool="same",
             seqs=48, min_keys=1, max_keys=4096, log_keys=False, heads=32, kv_heads=8,
             head_dim=128, block_size=32, lengths=5),
        # Chunked prefill of a mixed iteration: 512-token chunks behind cached prefixes.
        dict(name="prefill_chunks_bf16", kind="prefill", dtype="bfloat16", pool="same",
             seqs=16, min_query=512, max_query=512, min_prior=0, max_prior=2048, heads=32,
             kv_heads=8, head_dim=128, block_size=16, lengths=6),
        # Whole ragged prompts of a model served in fp32, its most exact setting (the
        # prompt lengths of the end-to-end workload).
        dict(name="prefill_prompts_fp32", kind="prefill", dtype="float32", pool="same",
             seqs=16, min_query=64, max_query=1024, min_prior=0, max_prior=0, heads=32,
             kv_heads=4, head_dim=64, block_size=16, lengths=7),
        # A few ragged chunks, odd ones among them, over fp8 pools.
        dict(name="prefill_ragged_fp8", kind="prefill", dtype="bfloat16", pool="fp8",
             seqs=5, min_query=1, max_query=777, min_prior=0, max_prior=4096, heads=32,
             kv_heads=8, head_dim=128, block_size=16, lengths=8),
        # RoPE and the KV append of a mixed iteration (16 chunks of 512 and 240 decodes).
        dict(name="append_rope_bf16", kind="append", dtype="bfloat16", pool="same",
             tokens=8432, heads=32, kv_heads=8, head_dim=128, block_size=16),
        # The residual add and norm between attention and MLP of a packed iteration.
        dict(name="norm_residual_bf16", kind="norm", dtype="bfloat16", rows=8627, hidden=4096),
        # Greedy choice for a small batch of running requests.
        dict(name="greedy_bf16", kind="greedy", dtype="bfloat16", rows=16, vocab=32000),
        # A whole iteration of the 1.1B model: three prompts and thirteen decodes.
        dict(name="model_iteration_bf16", kind="model", dtype="bfloat16", prompts=3,
             min_query=64, max_query=512, decodes=13, min_keys=64, max_keys=1024,
             block_size=16, lengths=9),
    ]


def _between(rng: random.Random, low: int, high: int) -> int:
    """An integer of [low, high], uniform over its logarithm."""

    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


# (query heads, KV heads, head_dim) of the layers served: the small fp32 layer, the 1.1B
# layer and the Llama-3-8B layer.
LAYERS = ((8, 2, 64), (32, 4, 64), (32, 8, 128))


def _draw_once(rng: random.Random) -> dict:
    kind = rng.choice(("decode", "decode", "decode", "prefill", "prefill", "append", "norm",
                       "greedy"))
    dtype = rng.choice(("bfloat16", "bfloat16", "float16", "float32"))
    heads, kv_heads, head_dim = rng.choice(LAYERS)
    layer = dict(heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                 block_size=rng.choice((16, 16, 32)))
    pool = rng.choice(("same", "same", "fp8", "fp8_rows"))
    lengths = rng.randrange(1 << 30)
    if kind == "decode":
        high = _between(rng, 64, 8192)
        return dict(kind=kind, fused=pool == "same" and rng.random() < 0.5, dtype=dtype, pool=pool,
                    seqs=_between(rng, 1, 256), min_keys=rng.randint(1, min(high, 128)),
                    max_keys=high, log_keys=rng.random() < 0.5, lengths=lengths, **layer)
    if kind == "prefill":
        high = _between(rng, 16, 1024)
        return dict(kind=kind, dtype=dtype, pool=pool, seqs=_between(rng, 1, 16),
                    min_query=rng.randint(1, high), max_query=high, min_prior=0,
                    max_prior=rng.choice((0, _between(rng, 16, 4096))), lengths=lengths, **layer)
    if kind == "append":
        return dict(kind=kind, dtype=dtype, pool="same", tokens=_between(rng, 1, 8432), **layer)
    if kind == "norm":
        return dict(kind=kind, dtype=dtype, rows=_between(rng, 1, 8627),
                    hidden=rng.choice((512, 2048, 4096)))
    return dict(kind=kind, dtype=dtype, rows=_between(rng, 1, 256),
                vocab=_between(rng, 1000, 131072))


def _cost(case: dict) -> tuple[float, float]:
    w = work(case)
    flops = w["flops"] if case["kind"] == "prefill" else 0.0
    return float(w["bytes"]), flops


def draw(rng: random.Random) -> dict:
    """A case of the listed ranges that costs no more than the listed one of its kind (and,
    for prefill, of its arithmetic: fp32 products or 16-bit ones)."""

    while True:
        case = _draw_once(rng)
        alike = [c for c in listed() if c["kind"] == case["kind"]
                 and (case["kind"] != "prefill"
                      or (c["dtype"] == "float32") == (case["dtype"] == "float32"))]
        size, flops = _cost(case)
        if (size <= max(_cost(c)[0] for c in listed() if c["kind"] == case["kind"])
                and flops <= max(_cost(c)[1] for c in alike)):
            return case


# ------------------------------------------------------------------ lengths


def _lengths(case: dict) -> list[int]:
    """Keys of each decode sequence (its new token's among them)."""

    rng = random.Random(case["lengths"])
    low, high = case["min_keys"], case["max_keys"]
    if case.get("log_keys"):
        return [_between(rng, low, high) for _ in range(case["seqs"])]
    return [rng.randint(low, high) for _ in range(case["seqs"])]


def _chunks(case: dict) -> list[tuple[int, int]]:
    """(query tokens, cached tokens before them) of each chunk."""

    rng = random.Random(case["lengths"])
    return [(rng.randint(case["min_query"], case["max_query"]),
             rng.randint(case["min_prior"], case["max_prior"])) for _ in range(case["seqs"])]


def _model_lengths(case: dict) -> tuple[list[int], list[int]]:
    rng = random.Random(case["lengths"])
    return ([rng.randint(case["min_query"], case["max_query"]) for _ in range(case["prompts"])],
            [rng.randint(case["min_keys"], case["max_keys"]) for _ in range(case["decodes"])])


def _causal_pairs(query: int, prior: int) -> int:
    return query * prior + query * (query + 1) // 2


# -------------------------------------------------------------------- work


def work(case: dict) -> dict:
    """Bytes (inputs read once, outputs written once) and operations of one pass."""

    kind = case["kind"]
    elem = 4 if case["dtype"] == "float32" else 2
    if kind == "norm":
        n = case["rows"] * case["hidden"]
        # input, residual, sum and normalised rows; the weight
        return {"bytes": 4 * n * elem + case["hidden"] * elem, "flops": 5 * n}
    if kind == "greedy":
        n = case["rows"] * case["vocab"]
        return {"bytes": n * elem + case["rows"] * 8, "flops": n}
    if kind == "model":
        cfg = tinyllama_1_1b()
        prompts, decodes = _model_lengths(case)
        tokens = sum(prompts) + len(decodes)
        d, i = cfg.hidden_size, cfg.intermediate_size
        kv = cfg.num_key_value_heads * cfg.head_dim
        layer = d * (2 * d + 2 * kv) + 3 * d * i
        head = cfg.vocab_size * d
        rows = len(prompts) + len(decodes)
        cached = sum(decodes) - len(decodes)
        pairs = sum(_causal_pairs(p, 0) for p in prompts) + sum(decodes)
        layers = cfg.num_hidden_layers
        return {"bytes": elem * (layers * (layer + 2 * kv * (cached + tokens)) + head
                                 + tokens * d + rows * cfg.vocab_size),
                "flops": 2 * layers * layer * tokens + 2 * rows * head
                + 4 * layers * pairs * d}
    row = case["head_dim"] * (elem if case["pool"] == "same" else 1)
    row += 4 if case["pool"] == "fp8_rows" else 0
    kv_row, q_row = 2 * case["kv_heads"] * row, case["heads"] * case["head_dim"] * elem
    if kind == "append":
        n = case["tokens"]
        new = 2 * case["kv_heads"] * case["head_dim"] * elem
        # query in and out, new rows in, pool rows out, position and slot; the table's rows
        return {"bytes": n * (2 * q_row + new + kv_row + 16 + case["head_dim"] * elem),
                "flops": 3 * n * (case["heads"] + case["kv_heads"]) * case["head_dim"]}
    if kind == "decode":
        keys = _lengths(case)
        size = sum(keys) * kv_row + 2 * len(keys) * q_row
        if case["fused"]:
            size += len(keys) * (2 * case["kv_heads"] * case["head_dim"] * elem + 16)
        return {"bytes": size, "flops": 4 * sum(keys) * case["heads"] * case["head_dim"]}
    chunks = _chunks(case)
    return {"bytes": sum((q + p) * kv_row + 2 * q * q_row for q, p in chunks),
            "flops": 4 * case["heads"] * case["head_dim"]
            * sum(_causal_pairs(q, p) for q, p in chunks)}


# ------------------------------------------------------------------ inputs


class _Values:
    """Seeded inputs, drawn on the device."""

    def __init__(self, seed: int) -> None:
        self.rng = torch.Generator(device=DEVICE).manual_seed(seed)
        self.host = torch.Generator().manual_seed(seed)

    def normal(self, *shape: int, dtype: torch.dtype = torch.float32) -> torch.Tensor:
        return torch.randn(shape, generator=self.rng, device=DEVICE).to(dtype)

    def uniform(self, *shape: int) -> torch.Tensor:
        return torch.rand(shape, generator=self.rng, device=DEVICE)

    def tables(self, counts: list[int]) -> tuple[torch.Tensor, int]:
        """Disjoint block tables (B, W) out of one random order of the pool's blocks."""

        total = sum(counts)
        order = torch.randperm(total, generator=self.host).to(torch.int32)
        tables = torch.zeros((len(counts), max(counts)), dtype=torch.int32)
        start = 0
        for b, count in enumerate(counts):
            tables[b, :count] = order[start:start + count]
            start += count
        return tables, total


def _pools(case: dict, values: _Values, blocks: int) -> dict:
    """K and V pools of one layer and the arguments that decode them."""

    shape = (1, blocks, case["kv_heads"], case["block_size"], case["head_dim"])
    keys, vals = values.normal(*shape), values.normal(*shape)
    if case["pool"] == "same":
        dtype = DTYPES[case["dtype"]]
        return {"key_cache": keys.to(dtype), "value_cache": vals.to(dtype), "scales": {}}
    if case["pool"] == "fp8":
        k, v = ((x / s).clamp(-448.0, 448.0).to(FP8) for x, s in zip((keys, vals), POOL_SCALES))
        return {"key_cache": k, "value_cache": v,
                "scales": {"k_scale": POOL_SCALES[0], "v_scale": POOL_SCALES[1]}}
    out: dict = {"scales": {}}
    for name, x in (("key", keys), ("value", vals)):
        x = x * torch.exp2(-6.0 * values.uniform(*shape[:4])).unsqueeze(-1)
        scale = x.abs().amax(dim=-1) / 448.0
        out[name + "_cache"] = (x / scale.unsqueeze(-1)).clamp(-448.0, 448.0).to(FP8)
        out["scales"][name[0] + "_scales"] = scale.contiguous()
    return out


def _attention_inputs(case: dict, seed: int, keys: list[int],
                      rows: int) -> tuple[dict, _Values]:
    values = _Values(seed)
    bs = case["block_size"]
    tables, blocks = values.tables([-(-n // bs) for n in keys])
    state = _pools(case, values, blocks)
    order = sorted(range(len(keys)), key=lambda b: (-keys[b], b))
    state.update(
        query=values.normal(rows, case["heads"], case["head_dim"], dtype=DTYPES[case["dtype"]]),
        block_tables=tables.to(DEVICE), host_tables=tables,
        seq_lens=torch.tensor(keys, dtype=torch.int32, device=DEVICE),
        seq_order=torch.tensor(order, dtype=torch.int32, device=DEVICE),
        max_seq_len=max(keys))
    return state, values


def _new_rows(case: dict, values: _Values, rows: int) -> dict:
    dtype = DTYPES[case["dtype"]]
    return {name: values.normal(rows, case["kv_heads"], case["head_dim"], dtype=dtype)
            for name in ("key", "value")}


def _decode_inputs(case: dict, seed: int) -> dict:
    keys = _lengths(case)
    state, values = _attention_inputs(case, seed, keys, len(keys))
    if case["fused"]:
        bs = case["block_size"]
        state.update(_new_rows(case, values, len(keys)))
        last = [n - 1 for n in keys]
        state["positions"] = torch.tensor(last, dtype=torch.int64, device=DEVICE)
        state["slots"] = torch.tensor(
            [int(state["host_tables"][b, p // bs]) * bs + p % bs for b, p in enumerate(last)],
            dtype=torch.int64, device=DEVICE)
    return state


def _prefill_inputs(case: dict, seed: int) -> dict:
    chunks = _chunks(case)
    state, _ = _attention_inputs(case, seed, [q + p for q, p in chunks], sum(q for q, _ in chunks))
    cu = [0]
    for q, _ in chunks:
        cu.append(cu[-1] + q)
    state["cu_seqlens_q"] = torch.tensor(cu, dtype=torch.int32, device=DEVICE)
    state["max_query_len"] = max(q for q, _ in chunks)
    return state


THETA = 500000.0
POSITIONS = 8192


def _append_inputs(case: dict, seed: int) -> dict:
    values = _Values(seed)
    n, bs, dtype = case["tokens"], case["block_size"], DTYPES[case["dtype"]]
    shape = (1, -(-n // bs), case["kv_heads"], bs, case["head_dim"])
    state = {"query": values.normal(n, case["heads"], case["head_dim"], dtype=dtype),
             "key_cache": torch.zeros(shape, dtype=dtype, device=DEVICE),
             "value_cache": torch.zeros(shape, dtype=dtype, device=DEVICE)}
    state.update(_new_rows(case, values, n))
    # Chunks of up to a block's tokens land in the blocks the allocator had free.
    blocks = torch.randperm(shape[1], generator=values.host)
    index = torch.arange(n)
    state["slots"] = (blocks[index // bs] * bs + index % bs).to(DEVICE)
    state["positions"] = torch.randint(0, POSITIONS, (n,), generator=values.host).to(DEVICE)
    return state


def _norm_inputs(case: dict, seed: int) -> dict:
    values = _Values(seed)
    dtype = DTYPES[case["dtype"]]
    shape = (case["rows"], case["hidden"])
    return {"inputs": values.normal(*shape, dtype=dtype),
            "residual": values.normal(*shape, dtype=dtype),
            "weight": (1.0 + 0.02 * values.normal(case["hidden"])).to(dtype)}


def _model_weights(seed: int, dtype: torch.dtype) -> dict:
    values = _Values(seed)
    cfg = tinyllama_1_1b()
    d, i, kv = cfg.hidden_size, cfg.intermediate_size, cfg.num_key_value_heads * cfg.head_dim

    def linear(out: int, into: int) -> torch.Tensor:
        return (values.normal(out, into) / math.sqrt(into)).to(dtype)

    def norm() -> torch.Tensor:
        return (1.0 + 0.02 * values.normal(d)).to(dtype)

    weights = {"embed_tokens.weight": values.normal(cfg.vocab_size, d, dtype=dtype)}
    for index in range(cfg.num_hidden_layers):
        at = f"layers.{index}."
        weights[at + "input_norm.weight"] = norm()
        for name, out in (("q", d), ("k", kv), ("v", kv), ("o", d)):
            weights[f"{at}self_attention.{name}_proj.weight"] = linear(out, d)
        weights[at + "post_attention_norm.weight"] = norm()
        weights[at + "mlp.gate_proj.weight"] = linear(i, d)
        weights[at + "mlp.up_proj.weight"] = linear(i, d)
        weights[at + "mlp.down_proj.weight"] = linear(d, i)
    weights["final_norm.weight"] = norm()
    weights["lm_head.weight"] = linear(cfg.vocab_size, d)
    return weights


def _model_inputs(case: dict, seed: int) -> dict:
    """Weights, token ids, block tables and the pools' cached rows."""

    cfg = tinyllama_1_1b()
    dtype = DTYPES[case["dtype"]]
    prompts, decodes = _model_lengths(case)
    weights = _model_weights(seed, dtype)
    values = _Values(seed + 1)
    bs = case["block_size"]
    tables, blocks = values.tables([-(-n // bs) for n in prompts + decodes])
    tokens = torch.randint(0, cfg.vocab_size, (sum(prompts) + len(decodes),),
                           generator=values.host)
    shape = (cfg.num_hidden_layers, blocks, cfg.num_key_value_heads, bs, cfg.head_dim)
    return {"weights": weights, "tables": tables, "blocks": blocks, "tokens": tokens,
            "keys": values.normal(*shape, dtype=dtype),
            "values": values.normal(*shape, dtype=dtype), "prompts": prompts, "decodes": decodes}


# ----------------------------------------------------------------- prepare


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "decode":
        state = _decode_inputs(case, seed)
        if case["fused"]:
            state["table"] = ops.RotaryTable(case["head_dim"], theta=THETA, max_position=POSITIONS,
                                             dtype=DTYPES[case["dtype"]], device=DEVICE)
        state["out"] = torch.empty_like(state["query"])
    elif kind == "prefill":
        state = _prefill_inputs(case, seed)
        state["out"] = torch.empty_like(state["query"])
    elif kind == "append":
        state = _append_inputs(case, seed)
        state["table"] = ops.RotaryTable(case["head_dim"], theta=THETA, max_position=POSITIONS,
                                         dtype=DTYPES[case["dtype"]], device=DEVICE)
        state["out"] = torch.empty_like(state["query"])
    elif kind == "norm":
        state = _norm_inputs(case, seed)
        state["sum"] = torch.empty_like(state["inputs"])
        state["out"] = torch.empty_like(state["inputs"])
    elif kind == "greedy":
        state = {"logits": 4.0 * _Values(seed).normal(case["rows"], case["vocab"])}
        state["logits"] = state["logits"].to(DTYPES[case["dtype"]])
    else:
        given = _model_inputs(case, seed)
        cfg = tinyllama_1_1b()
        with torch.device("meta"):
            model = LlamaModel(cfg)
        model.load_state_dict(given["weights"], assign=True)
        storage = PagedKVStorage(
            num_layers=cfg.num_hidden_layers, num_blocks=given["blocks"],
            num_key_value_heads=cfg.num_key_value_heads, block_size=case["block_size"],
            head_dim=cfg.head_dim, device=given["keys"].device, dtype=given["keys"].dtype)
        storage.key_storage.copy_(given["keys"])
        storage.value_storage.copy_(given["values"])
        model.rotary_table()
        works, start = [], 0
        for b, n in enumerate(given["prompts"] + given["decodes"]):
            count = n if b < len(given["prompts"]) else 1
            table = given["tables"][b, :-(-n // case["block_size"])].tolist()
            works.append(SequenceWork(given["tokens"][start:start + count].tolist(), n - count,
                                      table))
            start += count
        split = len(given["prompts"])
        batch = PackedBatchBuilder(given["keys"].device, case["block_size"]).build(
            works[:split], works[split:])
        state = {"model": model.eval(), "storage": storage, "batch": batch}
    state["case"] = case
    return state


# --------------------------------------------------------------------- run


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode" and case["fused"]:
        ops.rope_append_paged_decode(
            state["query"], state["key"], state["value"], state["positions"], state["table"],
            state["key_cache"], state["value_cache"], state["slots"], state["block_tables"],
            state["seq_lens"], layer_index=0, max_seq_len=state["max_seq_len"], out=state["out"],
            seq_order=state["seq_order"])
        return state["out"], state["key_cache"], state["value_cache"]
    if kind == "decode":
        return ops.paged_attention_decode(
            state["query"], state["key_cache"], state["value_cache"], state["block_tables"],
            state["seq_lens"], layer_index=0, max_seq_len=state["max_seq_len"], out=state["out"],
            seq_order=state["seq_order"], **state["scales"])
    if kind == "prefill":
        return ops.paged_attention_prefill(
            state["query"], state["key_cache"], state["value_cache"], state["block_tables"],
            state["seq_lens"], state["cu_seqlens_q"], layer_index=0,
            max_query_len=state["max_query_len"], max_seq_len=state["max_seq_len"],
            out=state["out"], seq_order=state["seq_order"], **state["scales"])
    if kind == "append":
        ops.rope_kv_append(state["query"], state["key"], state["value"], state["positions"],
                           state["table"], state["key_cache"], state["value_cache"],
                           state["slots"], 0, query_out=state["out"])
        return state["out"], state["key_cache"], state["value_cache"]
    if kind == "norm":
        return ops.rms_norm(state["inputs"], state["weight"], 1e-5, residual=state["residual"],
                            residual_out=state["sum"], out=state["out"]), state["sum"]
    if kind == "greedy":
        return ops.greedy_argmax(state["logits"])
    storage = state["storage"]
    logits = state["model"].forward_packed(state["batch"], storage)
    return logits, storage.key_storage, storage.value_storage


# --------------------------------------------------------------- tolerance


def tolerance(case: dict):
    """Largest difference of two correct results: about four times the distance measured
    between `run` and `exact` (fp32 sums; 16-bit roundings of inputs and results)."""

    kind = case["kind"]
    if kind == "greedy":
        return "exact"
    if kind == "model":
        return {"rel": 8e-2}
    if case["dtype"] == "float32":
        return {"rel": 2e-6}
    return {"rel": 1e-2 if case["dtype"] == "bfloat16" else 2e-3}


# ------------------------------------------------------------------- exact


def _rotary(head_dim: int, theta: float, dtype: torch.dtype) -> tuple[torch.Tensor, torch.Tensor]:
    """cos and sin rows as the model defines them: fp32 angles, rounded to its dtype."""

    inverse = theta ** (-torch.arange(0, head_dim, 2, dtype=torch.float32) / head_dim)
    angles = torch.outer(torch.arange(POSITIONS, dtype=torch.float32), inverse)
    return (angles.cos().to(dtype).to(DEVICE).double(), angles.sin().to(dtype).to(DEVICE).double())


def _rotate(x: torch.Tensor, positions: torch.Tensor, table) -> torch.Tensor:
    """x (N, H, Dh) in 64 bits rotated by halves at positions (N,)."""

    cos, sin = (t[positions].unsqueeze(1) for t in table)
    a, b = x.double().chunk(2, dim=-1)
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def _attend(query: torch.Tensor, keys: torch.Tensor, values: torch.Tensor) -> torch.Tensor:
    """query (T, Hq, Dh), the last T positions of keys and values (S, Hkv, Dh): causal."""

    t, hq, dh = query.shape
    s, hkv, _ = keys.shape
    g = hq // hkv
    q = query.view(t, hkv, g, dh).permute(1, 2, 0, 3).reshape(hkv, g * t, dh)
    scores = (q @ keys.permute(1, 2, 0).contiguous()).view(hkv, g, t, s) / math.sqrt(dh)
    hidden = torch.ones(t, s, dtype=torch.bool, device=query.device).triu(s - t + 1)
    probs = scores.masked_fill_(hidden, -math.inf).softmax(dim=-1).view(hkv, g * t, s)
    out = probs @ values.permute(1, 0, 2).contiguous()
    return out.view(hkv, g, t, dh).permute(2, 0, 1, 3).reshape(t, hq, dh)


def _decoded(state: dict) -> tuple[torch.Tensor, torch.Tensor]:
    """One layer's pools in 64 bits, (NB, Hkv, BS, Dh)."""

    pools = []
    for name in ("key", "value"):
        pool = state[name + "_cache"][0].to(torch.float32).double()
        scales = state["scales"]
        if name[0] + "_scales" in scales:
            pool = pool * scales[name[0] + "_scales"][0].double().unsqueeze(-1)
        elif scales:
            pool = pool * scales[name[0] + "_scale"]
        pools.append(pool)
    return pools[0], pools[1]


def _rows(pool: torch.Tensor, table: torch.Tensor, count: int) -> torch.Tensor:
    """The first `count` positions behind a block table, (count, Hkv, Dh)."""

    blocks = pool[table.long()]  # (n, Hkv, BS, Dh)
    return blocks.permute(0, 2, 1, 3).reshape(-1, pool.shape[1], pool.shape[3])[:count]


def _exact_model(case: dict, seed: int) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Logits and both pools after the iteration."""

    cfg = tinyllama_1_1b()
    given = _model_inputs(case, seed)
    weights = given["weights"]
    bs = case["block_size"]
    table = _rotary(cfg.head_dim, cfg.rope_theta, DTYPES[case["dtype"]])
    lengths = given["prompts"] + given["decodes"]
    counts = given["prompts"] + [1] * len(given["decodes"])
    positions = torch.cat([torch.arange(n - c, n) for n, c in zip(lengths, counts)]).to(DEVICE)

    def norm(x: torch.Tensor, name: str) -> torch.Tensor:
        scale = torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + cfg.rms_norm_eps)
        return x * scale * weights[name].double()

    def linear(x: torch.Tensor, name: str) -> torch.Tensor:
        return x @ weights[name].double().t()

    x = weights["embed_tokens.weight"][given["tokens"].to(DEVICE)].double()
    n = x.shape[0]
    pools = given["keys"].double(), given["values"].double()
    sequence = [b for b, c in enumerate(counts) for _ in range(c)]
    blocks = given["tables"][sequence, positions.cpu() // bs].long().to(DEVICE)
    offsets = positions % bs
    for index in range(cfg.num_hidden_layers):
        at = f"layers.{index}."
        h = norm(x, at + "input_norm.weight")
        q, k, v = (linear(h, f"{at}self_attention.{p}_proj.weight").view(n, -1, cfg.head_dim)
                   for p in "qkv")
        q, k = _rotate(q, positions, table), _rotate(k, positions, table)
        for pool, new in zip(pools, (k, v)):
            pool[index][blocks, :, offsets] = new
        out, start = [], 0
        for b, (length, count) in enumerate(zip(lengths, counts)):
            table_row = given["tables"][b, :-(-length // bs)].to(DEVICE)
            keys, vals = (_rows(pool[index], table_row, length) for pool in pools)
            out.append(_attend(q[start:start + count], keys, vals))
            start += count
        x = x + linear(torch.cat(out).reshape(n, -1), at + "self_attention.o_proj.weight")
        h = norm(x, at + "post_attention_norm.weight")
        gate = torch.nn.functional.silu(linear(h, at + "mlp.gate_proj.weight"))
        x = x + linear(gate * linear(h, at + "mlp.up_proj.weight"), at + "mlp.down_proj.weight")
    last = torch.tensor(counts).cumsum(0).to(DEVICE) - 1
    return (linear(norm(x[last], "final_norm.weight"), "lm_head.weight"), *pools)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "model":
        return _exact_model(case, seed)
    if kind == "greedy":
        return prepare(case, seed)["logits"].float().argmax(dim=-1, keepdim=True)
    if kind == "norm":
        state = _norm_inputs(case, seed)
        total = state["inputs"].double() + state["residual"].double()
        # The sum is a result in the rows' dtype; what is normalised is that result.
        x = total.to(DTYPES[case["dtype"]]).double()
        scale = torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + 1e-5)
        return x * scale * state["weight"].double(), total
    dtype = DTYPES[case["dtype"]]
    if kind == "append":
        state = _append_inputs(case, seed)
        table = _rotary(case["head_dim"], THETA, dtype)
        pools = [state[name + "_cache"].double() for name in ("key", "value")]
        blocks, rows = state["slots"] // case["block_size"], state["slots"] % case["block_size"]
        pools[0][0][blocks, :, rows] = _rotate(state["key"], state["positions"], table)
        pools[1][0][blocks, :, rows] = state["value"].double()
        return _rotate(state["query"], state["positions"], table), pools[0], pools[1]
    if kind == "decode":
        state = _decode_inputs(case, seed)
        lengths = _lengths(case)
        counts = [1] * len(lengths)
    else:
        state = _prefill_inputs(case, seed)
        lengths = [q + p for q, p in _chunks(case)]
        counts = [q for q, _ in _chunks(case)]
    query = state["query"].double()
    keys, vals = _decoded(state)
    fused = kind == "decode" and case["fused"]
    if fused:
        table = _rotary(case["head_dim"], THETA, dtype)
        query = _rotate(state["query"], state["positions"], table)
        blocks, rows = state["slots"] // case["block_size"], state["slots"] % case["block_size"]
        keys[blocks, :, rows] = _rotate(state["key"], state["positions"], table)
        vals[blocks, :, rows] = state["value"].double()
    out = torch.empty_like(query)
    start = 0
    for b, (length, count) in enumerate(zip(lengths, counts)):
        blocks = state["block_tables"][b, :-(-length // case["block_size"])]
        out[start:start + count] = _attend(query[start:start + count], _rows(keys, blocks, length),
                                           _rows(vals, blocks, length))
        start += count
    return (out, keys.unsqueeze(0), vals.unsqueeze(0)) if fused else out
