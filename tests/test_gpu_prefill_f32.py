"""fp32 prefill on the matrix cores against the oracle in 64 bits.

rtol 1e-5, atol 1e-6 as for every fp32 result (the parity contract); outputs here average
values of unit size, and each is a handful of chains of at most a few hundred fp32 sums.
"""

import pytest
import torch
from torch.testing import assert_close

from oracle import paged
from tokserve_amd import workloads
from tokserve_amd.kernels import ops

pytestmark = pytest.mark.gpu

TOL = dict(rtol=1e-5, atol=1e-6)
POOL_SCALES = dict(k_scale=0.5, v_scale=0.25)


def _run(batch, keys, values, **scales):
    out = ops.paged_attention_prefill(
        batch.query, keys, values, batch.block_tables, batch.seq_lens, batch.cu_seqlens_q,
        layer_index=0, max_query_len=batch.max_query_len, max_seq_len=batch.max_seq_len, **scales)
    torch.cuda.synchronize()
    return out.cpu()


def _oracle(batch, keys, values):
    return paged.prefill_batch(batch.query.cpu(), keys, values, batch.block_tables.cpu(),
                               batch.seq_lens.cpu(), batch.cu_seqlens_q.cpu(), 0, torch.float64)


# Contexts and chunks around a step's 32 keys, a page and a tile of 128 / G query tokens.
CONTEXTS, CHUNKS = [1, 32, 33, 64, 65, 200, 300, 77], [1, 32, 33, 17, 64, 129, 1, 16]


@pytest.mark.parametrize("pool", ["same", "fp8", "fp8_rows"])
@pytest.mark.parametrize(("hq", "hkv", "dh", "block_size"),
                         [(32, 4, 64, 16), (8, 2, 128, 32), (2, 2, 128, 16), (16, 1, 64, 16),
                          (6, 2, 64, 7), (5, 1, 128, 48)])
def test_prefill_f32_shapes(device, hq, hkv, dh, block_size, pool) -> None:
    batch = workloads.paged_batch(CONTEXTS, CHUNKS, num_q_heads=hq, num_kv_heads=hkv, head_dim=dh,
                                  block_size=block_size, dtype=torch.float32, device=device,
                                  seed=dh + hq)
    keys, values = batch.key_cache.cpu(), batch.value_cache.cpu()
    if pool == "same":
        got = _run(batch, batch.key_cache, batch.value_cache)
    elif pool == "fp8":
        k8 = paged.quantize_e4m3(keys, POOL_SCALES["k_scale"])
        v8 = paged.quantize_e4m3(values, POOL_SCALES["v_scale"])
        got = _run(batch, k8.to(device), v8.to(device), **POOL_SCALES)
        keys = paged.dequantize_e4m3(k8, POOL_SCALES["k_scale"], torch.float32)
        values = paged.dequantize_e4m3(v8, POOL_SCALES["v_scale"], torch.float32)
    else:
        (k8, ks), (v8, vs) = paged.quantize_e4m3_rows(keys), paged.quantize_e4m3_rows(values)
        got = _run(batch, k8.to(device), v8.to(device), k_scales=ks.to(device),
                   v_scales=vs.to(device))
        keys = paged.dequantize_e4m3_rows(k8, ks, torch.float64)
        values = paged.dequantize_e4m3_rows(v8, vs, torch.float64)
    assert_close(got, _oracle(batch, keys, values), **TOL)


@pytest.mark.parametrize(("hq", "hkv"), [(8, 2), (32, 4)])
def test_prefill_f32_strided_rows_and_moving_reference(device, hq, hkv) -> None:
    """Query and output rows inside wider ones, and keys that grow along each sequence, so
    that the softmax reference moves many times: few rows (on the VALU kernel) and more."""

    batch = workloads.paged_batch([700, 40], [200, 40], num_q_heads=hq, num_kv_heads=hkv,
                                  head_dim=64, block_size=16, dtype=torch.float32, device=device,
                                  seed=3)
    for b, context in enumerate([700, 40]):
        for i in range((context + 15) // 16):
            batch.key_cache[0, int(batch.block_tables[b, i])] *= 1 + i / 8
    wide = torch.zeros(240, hq, 72, device=device)
    wide[..., :64] = batch.query
    out = torch.full((240, hq + 4, 64), 7.0, device=device)
    ops.paged_attention_prefill(
        wide[..., :64], batch.key_cache, batch.value_cache, batch.block_tables, batch.seq_lens,
        batch.cu_seqlens_q, layer_index=0, max_query_len=200, max_seq_len=700, out=out[:, :hq])
    torch.cuda.synchronize()
    expected = _oracle(batch, batch.key_cache.cpu(), batch.value_cache.cpu())
    # Scores reach ~30 here, where one fp32 rounding is up to 2^-20; a sum of Dh products
    # gathers about sqrt(Dh) = 8 of them, so an exponent is off by up to 8e-6 and an output
    # by twice that times the largest |v| (~4).
    assert_close(out[:, :hq].cpu(), expected, rtol=0, atol=6e-5)
    assert bool((out[:, hq:] == 7.0).all())


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_prefill_f32_values_past_a_row_do_not_reach_it(device, dh, bad) -> None:
    """A value that is not finite reaches the rows that see its key and no other."""

    batch = workloads.paged_batch([100, 90], [60, 90], num_q_heads=4, num_kv_heads=1, head_dim=dh,
                                  block_size=16, dtype=torch.float32, device=device, seed=5)
    clean = _oracle(batch, batch.key_cache.cpu(), batch.value_cache.cpu())
    key = 70  # query token 30 of the first chunk
    batch.value_cache[0, int(batch.block_tables[0, key // 16]), 0, key % 16, dh - 3] = bad
    got = _run(batch, batch.key_cache, batch.value_cache)
    hit = torch.zeros_like(got, dtype=torch.bool)
    hit[30:60, :, dh - 3] = True
    assert not bool(got[hit].isfinite().any())
    assert_close(got[~hit], clean[~hit], **TOL)


@pytest.mark.parametrize("pool", ["same", "fp8_rows"])
@pytest.mark.parametrize(("contexts", "chunks", "layer"), [
    ([496, 90], [20, 28], (32, 8, 128)), ([512, 90], [20, 28], (32, 8, 128)),
    ([600, 90], [20, 29], (32, 8, 128)), ([112, 90], [9, 11], (32, 8, 128)),
    ([128, 90], [9, 11], (32, 8, 128)), ([128, 90], [10, 11], (32, 8, 128)),
    ([4000, 90], [60, 44], (32, 4, 64)), ([4000, 90], [60, 45], (32, 4, 64)),
    ([3980, 90], [60, 44], (32, 4, 64))])
def test_prefill_f32_few_rows_over_many_keys(device, contexts, chunks, layer, pool) -> None:
    """Both sides of the rules that leave few rows over many keys to the VALU kernel: 48 and 49
    tokens of 32 heads x 128 below and from 512 keys, 20 and 21 from 128 (fp32 pools), 104 and
    105 of 32 heads x 64 from 4,000."""

    kw = dict(kv_dtype=torch.float8_e4m3fn, scale_granularity="row") if pool != "same" else {}
    hq, hkv, dh = layer
    batch = workloads.paged_batch(contexts, chunks, num_q_heads=hq, num_kv_heads=hkv, head_dim=dh,
                                  block_size=16, dtype=torch.float32, device=device, seed=6, **kw)
    got = _run(batch, batch.key_cache, batch.value_cache, **batch.scale_kwargs)
    pools = []
    for cache, scales in ((batch.key_cache, batch.k_scales), (batch.value_cache, batch.v_scales)):
        rows = cache.cpu().double()
        pools.append(rows if scales is None else rows * scales.cpu().double().unsqueeze(-1))
    assert_close(got, _oracle(batch, *pools), **TOL)


def test_prefill_f32_more_workgroups_than_a_launch_holds(device) -> None:
    """2,048 chunks of four tokens under a bound of 8,192, 16 KV heads: a tile for every
    sequence, KV head and 16 tokens of the bound are 2^24 workgroups, 2^32 threads, one more
    than a launch may have. The VALU kernel, a workgroup per token, takes them."""

    seqs, hq, hkv, dh = 2048, 64, 16, 64
    batch = workloads.paged_batch([4 + i % 29 for i in range(seqs)], [4] * seqs, num_q_heads=hq,
                                  num_kv_heads=hkv, head_dim=dh, block_size=16,
                                  dtype=torch.float32, device=device, seed=8,
                                  pool_on_device_rng=True)
    tables = torch.zeros((seqs, 512), dtype=torch.int32, device=device)
    tables[:, :batch.block_tables.shape[1]] = batch.block_tables
    out = ops.paged_attention_prefill(
        batch.query, batch.key_cache, batch.value_cache, tables, batch.seq_lens,
        batch.cu_seqlens_q, layer_index=0, max_query_len=8192, max_seq_len=8192)
    # (the same chunks 64 at a time, which the other work order takes)
    for first in range(0, seqs, 64 * 8):
        part = slice(first, first + 64)
        rows = slice(4 * first, 4 * (first + 64))
        expected = ops.paged_attention_prefill(
            batch.query[rows], batch.key_cache, batch.value_cache, batch.block_tables[part],
            batch.seq_lens[part], batch.cu_seqlens_q[first:first + 65] - 4 * first, layer_index=0,
            max_query_len=4, max_seq_len=32)
        assert_close(out[rows], expected, **TOL)


@pytest.mark.parametrize("pool", ["same", "fp8_rows"])
@pytest.mark.parametrize("seqs", [64, 65, 100])
def test_prefill_f32_many_sequences(device, seqs, pool) -> None:
    """Up to 64 sequences the tiles are found in the order of their keys, past that level by
    level: empty chunks, chunks of one and of several tiles, with and without an order."""

    chunks = [(0, 1, 17, 40, 5, 130, 16)[i % 7] for i in range(seqs)]
    contexts = [q + (0, 3, 250, 31)[i % 4] for i, q in enumerate(chunks)]
    kw = dict(kv_dtype=torch.float8_e4m3fn, scale_granularity="row") if pool != "same" else {}
    batch = workloads.paged_batch(contexts, chunks, num_q_heads=8, num_kv_heads=2, head_dim=64,
                                  block_size=16, dtype=torch.float32, device=device, seed=seqs,
                                  **kw)
    pools = []
    for cache, scales in ((batch.key_cache, batch.k_scales), (batch.value_cache, batch.v_scales)):
        rows = cache.cpu().double()
        pools.append(rows if scales is None else rows * scales.cpu().double().unsqueeze(-1))
    expected = _oracle(batch, *pools)
    for order in (None, ops.longest_first(contexts, device)):
        got = _run(batch, batch.key_cache, batch.value_cache, seq_order=order,
                   **batch.scale_kwargs)
        assert_close(got, expected, **TOL)


@pytest.mark.parametrize("pool", ["fp8", "fp8_rows"])
@pytest.mark.parametrize(("hq", "dh"), [(8, 64), (2, 128), (16, 128)])
def test_prefill_f32_codes_past_a_row_do_not_reach_it(device, hq, dh, pool) -> None:
    """The same over e4m3 pools: a NaN code reaches its dimension of the rows that see its key,
    an infinite row scale every dimension of them, and no other row."""

    kw = (dict(k_scale=0.5, v_scale=0.25) if pool == "fp8" else dict(scale_granularity="row"))
    batch = workloads.paged_batch([100, 90], [60, 90], num_q_heads=hq, num_kv_heads=1, head_dim=dh,
                                  block_size=16, dtype=torch.float32, device=device, seed=5,
                                  kv_dtype=torch.float8_e4m3fn, **kw)
    pools = []
    for cache, scale, scales in ((batch.key_cache, batch.k_scale, batch.k_scales),
                                 (batch.value_cache, batch.v_scale, batch.v_scales)):
        rows = cache.cpu().double()
        pools.append(rows * (scale if scales is None else scales.cpu().double().unsqueeze(-1)))
    clean = _oracle(batch, *pools)
    key = 70  # query token 30 of the first chunk
    at = (0, int(batch.block_tables[0, key // 16]), 0, key % 16)
    hit = torch.zeros(clean.shape, dtype=torch.bool)
    if pool == "fp8":
        batch.value_cache.view(torch.uint8)[(*at, dh - 3)] = 0x7F
        hit[30:60, :, dh - 3] = True
    else:
        batch.v_scales[at] = float("inf")
        hit[30:60] = True
    got = _run(batch, batch.key_cache, batch.value_cache, **batch.scale_kwargs)
    assert not bool(got[hit].isfinite().any())
    assert_close(got[~hit], clean[~hit], **TOL)
