"""fp32 decode on the matrix cores against the oracle in 64 bits, at the edges of pages,
blocks and key splits, and the fused step against its two calls, bit for bit.

rtol 1e-5, atol 1e-6 as for every fp32 result (the parity contract).
"""

import pytest
import torch
from torch.testing import assert_close

from oracle import paged
from tests.test_gpu_fused_decode import _inputs
from tokserve_amd import workloads
from tokserve_amd.kernels import ops

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
TOL = dict(rtol=1e-5, atol=1e-6)
CONTEXTS = [1, 15, 16, 17, 0, 33, 128, 129, 400, 1000]


def _batch(device, contexts, hq, hkv, dh, block_size, pool):
    kw = {"same": {}, "fp8": dict(kv_dtype=FP8, k_scale=0.5, v_scale=0.25),
          "fp8_rows": dict(kv_dtype=FP8, scale_granularity="row")}[pool]
    return workloads.paged_batch(contexts, [1] * len(contexts), num_q_heads=hq, num_kv_heads=hkv,
                                 head_dim=dh, block_size=block_size, dtype=torch.float32,
                                 device=device, seed=hq + dh, **kw)


def _poison(batch, pool):
    """NaN in the rows past each sequence's last key: they must not reach a result."""

    block_size = batch.key_cache.shape[3]
    tables = batch.block_tables.cpu()
    for b, n in enumerate(batch.contexts):
        if n % block_size:
            block = int(tables[b, n // block_size])
            for cache in (batch.key_cache, batch.value_cache):
                rows = cache[0, block, :, n % block_size:]
                if pool == "same":
                    rows.fill_(float("nan"))
                else:
                    rows.view(torch.uint8).fill_(0x7F)
            if pool == "fp8_rows":
                for scales in (batch.k_scales, batch.v_scales):
                    scales[0, block, :, n % block_size:] = float("nan")


def _oracle(batch):
    pools = []
    for cache, scale, scales in ((batch.key_cache, batch.k_scale, batch.k_scales),
                                 (batch.value_cache, batch.v_scale, batch.v_scales)):
        pool = cache.cpu().double()
        pools.append(pool * (scale if scales is None else scales.cpu().double().unsqueeze(-1)))
    return paged.decode_batch(batch.query.cpu(), pools[0], pools[1], batch.block_tables.cpu(),
                              batch.seq_lens.cpu(), 0, torch.float64)


@pytest.mark.parametrize("pool", ["same", "fp8", "fp8_rows"])
@pytest.mark.parametrize(("hq", "hkv", "dh", "block_size"),
                         [(8, 2, 64, 16), (32, 8, 128, 16), (32, 4, 64, 48), (3, 1, 128, 32),
                          (16, 1, 128, 16), (2, 2, 64, 16)])
def test_decode_f32_shapes(device, hq, hkv, dh, block_size, pool) -> None:
    batch = _batch(device, CONTEXTS, hq, hkv, dh, block_size, pool)
    expected = _oracle(batch)
    _poison(batch, pool)
    order = ops.longest_first(batch.contexts, device)
    # Unsplit (8 waves), splits of one and three blocks, unsplit with 4 waves, and a host
    # bound past the lengths for which the library splits.
    for kw in (dict(), dict(pages_per_split=1), dict(pages_per_split=3, seq_order=order),
               dict(pages_per_split=1000), dict(max_seq_len=1040)):
        args = dict(layer_index=0, max_seq_len=batch.max_seq_len, **batch.scale_kwargs) | kw
        if args["max_seq_len"] > batch.block_tables.shape[1] * block_size:
            continue
        out = ops.paged_attention_decode(batch.query, batch.key_cache, batch.value_cache,
                                         batch.block_tables, batch.seq_lens, **args)
        torch.cuda.synchronize()
        assert_close(out.cpu(), expected, **TOL)


def test_decode_f32_many_and_long_sequences(device) -> None:
    """More than 64 pages per wave (page ids come 64 at a time), and a batch of more (sequence,
    KV head) pairs than CUs."""

    batch = _batch(device, [8200, 3, 4097], 4, 1, 64, 16, "same")
    for kw in (dict(), dict(pages_per_split=513)):
        out = ops.paged_attention_decode(batch.query, batch.key_cache, batch.value_cache,
                                         batch.block_tables, batch.seq_lens, layer_index=0,
                                         max_seq_len=batch.max_seq_len, **kw)
        torch.cuda.synchronize()
        assert_close(out.cpu(), _oracle(batch), **TOL)
    batch = _batch(device, [1 + (i * 37) % 300 for i in range(160)], 8, 2, 128, 16, "same")
    out = ops.paged_attention_decode(batch.query, batch.key_cache, batch.value_cache,
                                     batch.block_tables, batch.seq_lens, layer_index=0,
                                     max_seq_len=batch.max_seq_len)
    torch.cuda.synchronize()
    assert_close(out.cpu(), _oracle(batch), **TOL)


@pytest.mark.parametrize(("hq", "hkv", "dh", "block_size"),
                         [(8, 2, 64, 16), (32, 8, 128, 32), (3, 1, 128, 16), (16, 1, 64, 48)])
@pytest.mark.parametrize("pages_per_split", [0, 2])
def test_decode_f32_fused_step_equals_its_two_calls(device, hq, hkv, dh, block_size,
                                                    pages_per_split) -> None:
    contexts = [1, 16, 17, 32, 513, 48, 49]
    batch, query, key, value, positions, slots, table = _inputs(
        device, torch.float32, hq, hkv, dh, contexts, seed=dh + hq, block_size=block_size)
    slots[3] = -1  # appends nothing: the pool's own row is attended to
    k_ref, v_ref, q_ref = batch.key_cache.clone(), batch.value_cache.clone(), query.clone()
    args = dict(layer_index=0, max_seq_len=batch.max_seq_len, pages_per_split=pages_per_split)
    ops.rope_kv_append(q_ref, key, value, positions, table, k_ref, v_ref, slots, 0)
    expected = ops.paged_attention_decode(q_ref, k_ref, v_ref, batch.block_tables, batch.seq_lens,
                                          **args)
    out = ops.rope_append_paged_decode(query, key, value, positions, table, batch.key_cache,
                                       batch.value_cache, slots, batch.block_tables,
                                       batch.seq_lens, **args)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int32), expected.view(torch.int32))
    assert torch.equal(batch.key_cache, k_ref) and torch.equal(batch.value_cache, v_ref)


@pytest.mark.parametrize("pool", ["same", "fp8_rows"])
@pytest.mark.parametrize(("dh", "hkv", "seqs", "keys"), [
    (64, 2, 8, 640), (64, 2, 8, 641), (128, 8, 3, 384), (128, 8, 3, 385), (128, 8, 16, 640),
    (128, 8, 17, 640), (128, 8, 17, 641)])
def test_decode_f32_unsplit_or_split(device, dh, hkv, seqs, keys, pool) -> None:
    """Both sides of the lines up to which a small batch runs unsplit (8 waves to a pair)."""

    contexts = [keys] + [1 + (37 * i) % keys for i in range(seqs - 1)]
    batch = _batch(device, contexts, 4 * hkv, hkv, dh, 16, pool)
    expected = _oracle(batch)
    _poison(batch, pool)
    out = ops.paged_attention_decode(batch.query, batch.key_cache, batch.value_cache,
                                     batch.block_tables, batch.seq_lens, layer_index=0,
                                     max_seq_len=keys, **batch.scale_kwargs)
    torch.cuda.synchronize()
    assert_close(out.cpu(), expected, **TOL)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize(("hq", "dh"), [(8, 64), (6, 128)])
def test_decode_f32_values_that_are_not_finite(device, hq, dh, bad) -> None:
    """A value that is not finite under a visible key reaches its dimension of that sequence and
    KV head as it is, and no other result, wherever the key lies among waves and splits."""

    contexts = [400, 400, 33]
    batch = _batch(device, contexts, hq, 2, dh, 16, "same")
    clean = _oracle(batch)
    group = hq // 2
    hit = torch.zeros(clean.shape, dtype=torch.bool)
    for b, key, head, dim in ((0, 5, 0, 3), (0, 399, 0, dh - 1), (1, 200, 1, 17), (2, 32, 1, 0)):
        block = int(batch.block_tables[b, key // 16])
        batch.value_cache[0, block, head, key % 16, dim] = bad
        hit[b, head * group:(head + 1) * group, dim] = True
    for pages_per_split in (0, 1, 3, 1000):
        out = ops.paged_attention_decode(batch.query, batch.key_cache, batch.value_cache,
                                         batch.block_tables, batch.seq_lens, layer_index=0,
                                         max_seq_len=400, pages_per_split=pages_per_split).cpu()
        assert_close(out[hit], torch.full_like(out[hit], bad), rtol=0, atol=0, equal_nan=True)
        assert_close(out[~hit], clean[~hit], **TOL)
