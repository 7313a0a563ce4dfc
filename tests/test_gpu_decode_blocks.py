"""Decode over blocks of several 16-token pages (the MFMA decode keeps page ids there, and
its probabilities at 24 bits) against the fp32 oracle, and the fused step against its two
calls, bit for bit.

Tolerance against the oracle: the result's one rounding to the stored dtype (half a step,
2^-9 relative for bf16, 2^-12 for fp16), doubled for values next to a power of two, and
2e-5 absolute for fp32 sums of up to 700 products of N(0, 1) values in another order.
"""

import pytest
import torch
from torch.testing import assert_close

from oracle import paged
from tokserve_amd import workloads
from tokserve_amd.kernels import ops

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
ROUNDING = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
CONTEXTS = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 95, 96, 97, 700]


def _batch(device, dtype, group, dh, block_size, pool, seed=3):
    kw = {"pool": {}, "fp8": dict(kv_dtype=FP8, k_scale=0.5, v_scale=0.25),
          "rows": dict(kv_dtype=FP8, scale_granularity="row")}[pool]
    batch = workloads.paged_batch(CONTEXTS, [1] * len(CONTEXTS), num_q_heads=2 * group,
                                  num_kv_heads=2, head_dim=dh, block_size=block_size, dtype=dtype,
                                  device=device, seed=seed, **kw)
    # Rows past each sequence's last key hold NaN: they must not reach a result.
    tables = batch.block_tables.cpu()
    for b, n in enumerate(CONTEXTS):
        if n % block_size:
            block = int(tables[b, n // block_size])
            for cache in (batch.key_cache, batch.value_cache):
                rows = cache[0, block, :, n % block_size:]
                if pool == "pool":
                    rows.fill_(float("nan"))
                else:
                    rows.view(torch.uint8).fill_(0x7F)  # e4m3 NaN
            if pool == "rows":
                for scales in (batch.k_scales, batch.v_scales):
                    scales[0, block, :, n % block_size:] = float("nan")
    return batch


def _decode(batch, query=None, **kw):
    return ops.paged_attention_decode(
        batch.query if query is None else query, batch.key_cache, batch.value_cache,
        batch.block_tables, batch.seq_lens, layer_index=0, max_seq_len=batch.max_seq_len,
        **batch.scale_kwargs, **kw)


def _oracle(batch):
    pools = []
    for cache, scale, scales in ((batch.key_cache, batch.k_scale, batch.k_scales),
                                 (batch.value_cache, batch.v_scale, batch.v_scales)):
        pool = cache.cpu().float()
        pools.append(pool * (scale if scales is None else scales.cpu().unsqueeze(-1)))
    return paged.decode_batch(batch.query.cpu().float(), *pools, batch.block_tables.cpu(),
                              batch.seq_lens.cpu(), 0, torch.float32)


@pytest.mark.parametrize("pool", ["pool", "fp8", "rows"])
@pytest.mark.parametrize(("dtype", "group", "dh", "block_size"), [
    (torch.bfloat16, 4, 128, 32), (torch.float16, 8, 64, 32), (torch.bfloat16, 2, 64, 48),
    (torch.float16, 1, 128, 256)])
def test_long_blocks_match_the_oracle(device, dtype, group, dh, block_size, pool) -> None:
    batch = _batch(device, dtype, group, dh, block_size, pool)
    expected = _oracle(batch)
    for pages_per_split in (0, 1, 3):
        out = _decode(batch, pages_per_split=pages_per_split).cpu()
        assert_close(out.float(), expected, rtol=ROUNDING[dtype], atol=2e-5)


def test_infinite_values_stay_infinite(device) -> None:
    """An infinite value in V reaches its dimension as an infinity, not as NaN."""

    batch = _batch(device, torch.bfloat16, 4, 128, 32, "pool")
    block = int(batch.block_tables[4, 0])
    batch.value_cache[0, block, :, 3, 5] = float("inf")
    out = _decode(batch).cpu()
    assert_close(out.float(), _oracle(batch), rtol=ROUNDING[torch.bfloat16], atol=2e-5)
    assert torch.isinf(out[4, :, 5]).all()


@pytest.mark.parametrize("pool", ["pool", "fp8", "rows"])
def test_fused_step_over_long_blocks_equals_its_two_calls(device, pool) -> None:
    dtype, dh, bs = torch.bfloat16, 64, 48
    batch = _batch(device, dtype, 4, dh, bs, pool)
    gen = torch.Generator().manual_seed(9)
    n = len(CONTEXTS)
    query, key, value = (torch.randn(n, h, dh, generator=gen).to(dtype).to(device)
                         for h in (8, 2, 2))
    tables = batch.block_tables.cpu()
    slots = torch.tensor([int(tables[b, (c - 1) // bs]) * bs + (c - 1) % bs
                          for b, c in enumerate(CONTEXTS)], dtype=torch.int64)
    slots[2] = -1  # appends nothing
    slots = slots.to(device)
    positions = (batch.seq_lens - 1).long()
    table = ops.RotaryTable(dh, theta=1e4, max_position=1024, dtype=dtype, device=device)

    def pools():
        kw = dict(batch.scale_kwargs)
        if pool == "rows":
            kw = {name: scales.clone() for name, scales in kw.items()}
        return [batch.key_cache.clone(), batch.value_cache.clone()], kw

    for pages_per_split in (0, 2):
        (kc, vc), kw = pools()
        q_ref = query.clone()
        ops.rope_kv_append(q_ref, key, value, positions, table, kc, vc, slots, 0, **kw)
        expected = ops.paged_attention_decode(q_ref, kc, vc, batch.block_tables, batch.seq_lens,
                                              layer_index=0, max_seq_len=batch.max_seq_len,
                                              pages_per_split=pages_per_split, **kw)
        (kc2, vc2), kw2 = pools()
        actual = ops.rope_append_paged_decode(
            query, key, value, positions, table, kc2, vc2, slots, batch.block_tables,
            batch.seq_lens, layer_index=0, max_seq_len=batch.max_seq_len,
            pages_per_split=pages_per_split, **kw2)
        assert torch.equal(actual.view(torch.int16).cpu(), expected.view(torch.int16).cpu())
        for a, b in ((kc, kc2), (vc, vc2)):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
        if pool == "rows":
            for name in kw:
                assert torch.equal(kw[name].nan_to_num(-1.0), kw2[name].nan_to_num(-1.0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_infinite_values_past_a_waves_first_page_ids(device, dtype) -> None:
    """An infinite value among more pages than a wave holds ids of at once (64): the wave
    takes all of its pages again. Rounding as above; 1e-4 absolute for sums of 9,000 keys."""

    batch = workloads.paged_batch([9000, 40], [1, 1], num_q_heads=8, num_kv_heads=2, head_dim=64,
                                  block_size=32, dtype=dtype, device=device, seed=4)
    for key in (5, 8990):
        block = int(batch.block_tables[0, key // 32])
        batch.value_cache[0, block, :, key % 32, key % 64] = float("inf")
    out = _decode(batch, pages_per_split=1000).cpu()
    assert_close(out.float(), _oracle(batch), rtol=ROUNDING[dtype], atol=1e-4)
    assert torch.isinf(out[0, :, [5, 8990 % 64]]).all()


@pytest.mark.parametrize("pool", ["pool", "fp8"])
@pytest.mark.parametrize(("dtype", "dh"), [(torch.float16, 64), (torch.float16, 128),
                                           (torch.bfloat16, 128)])
def test_small_probabilities_keep_their_bits(device, dtype, dh, pool) -> None:
    """One key of each page holds nearly all of the weight and a value of 0; the other keys, of
    about e^-18 (2^-26) each, make up the whole result. An fp32 exponent of up to 27 is within
    2^-19 relative, so the result's one rounding is all that shows."""

    kw = dict(kv_dtype=FP8, k_scale=1.0, v_scale=16.0) if pool == "fp8" else {}
    batch = workloads.paged_batch([8192, 1000], [1, 1], num_q_heads=8, num_kv_heads=2,
                                  head_dim=dh, block_size=32, dtype=dtype, device=device, seed=6,
                                  **kw)
    top = (torch.arange(32, device=device) % 16 == 0)[:, None]
    size = 1.125 if dh == 64 else 0.8125  # scores of -9 and 9, or about
    batch.query.fill_(1.0)
    batch.key_cache.copy_(torch.where(top, size, -size).expand(batch.key_cache.shape))
    gen = torch.Generator().manual_seed(1)
    values = 200 + 240 * torch.rand(batch.value_cache.shape, generator=gen).to(device)
    batch.value_cache.copy_(torch.where(top, 0.0, values if pool == "fp8" else 16 * values))
    pools = [cache.cpu().double() * scale for cache, scale in
             ((batch.key_cache, batch.k_scale), (batch.value_cache, batch.v_scale))]
    expected = paged.decode_batch(batch.query.cpu().double(), *pools, batch.block_tables.cpu(),
                                  batch.seq_lens.cpu(), 0, torch.float64)
    for pages_per_split in (0, 1000):
        out = _decode(batch, pages_per_split=pages_per_split).cpu()
        assert_close(out.double(), expected, rtol=ROUNDING[dtype], atol=0)
