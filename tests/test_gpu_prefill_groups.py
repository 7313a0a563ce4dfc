"""bf16/fp16 prefill of few tiles: 64-row tiles and two groups of waves per tile, on both
sides of the rules that choose them, against the fp32 oracle.

Tolerance as for every 16-bit result: 2e-2 absolute of the reference kernel's fp32
arithmetic (plus one step of the stored dtype for the few-key rows with |o| past 2).
"""

import pytest
import torch
from torch.testing import assert_close

from oracle import paged
from tokserve_amd import workloads
from tokserve_amd.kernels import ops

pytestmark = pytest.mark.gpu

# (contexts, chunks): one key, a step's 32 keys and one more (the second group has none, or
# one, of them), odd and even step counts, tiles of one token; up to 255, 256 and more keys.
SMALL = ([1, 32, 33, 64, 65, 97, 200], [1, 32, 33, 64, 1, 97, 17])
HALF = (SMALL[0] + [256, 300], SMALL[1] + [256, 129])
# 257 to 512 tiles of 128 rows (32 / 8 heads at Dh 128, 32 / 4 at Dh 64), with a table of
# 1,024 keys or just below.
MIDDLE = ([1100, 300, 33, 700, 65], [300, 300, 33, 290, 65])
SHORTER = ([1000, 300, 33, 700, 65], [300, 300, 33, 290, 65])


def _check(device, dtype, hq, hkv, dh, lengths, block_size=16, **kw):
    batch = workloads.paged_batch(lengths[0], lengths[1], num_q_heads=hq, num_kv_heads=hkv,
                                  head_dim=dh, block_size=block_size, dtype=dtype, device=device,
                                  seed=dh + hq)
    out = ops.paged_attention_prefill(
        batch.query, batch.key_cache, batch.value_cache, batch.block_tables, batch.seq_lens,
        batch.cu_seqlens_q, layer_index=0, max_query_len=batch.max_query_len,
        max_seq_len=batch.max_seq_len, **kw)
    torch.cuda.synchronize()
    expected = paged.prefill_batch(
        batch.query.cpu(), batch.key_cache.cpu(), batch.value_cache.cpu(),
        batch.block_tables.cpu(), batch.seq_lens.cpu(), batch.cu_seqlens_q.cpu(), 0,
        torch.float32)
    assert_close(out.cpu(), expected, rtol=2.0 ** -7, atol=2e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("hq", "hkv", "dh"),
                         [(32, 8, 128), (32, 4, 64), (2, 2, 128), (2, 1, 64), (16, 1, 64),
                          (8, 1, 128), (16, 1, 128), (4, 2, 128)])
@pytest.mark.parametrize("lengths", [SMALL, HALF])
def test_prefill_half_tiles(device, dtype, hq, hkv, dh, lengths) -> None:
    _check(device, dtype, hq, hkv, dh, lengths, block_size=32 if hkv == 1 else 16)


@pytest.mark.parametrize(("hq", "hkv", "dh"), [(32, 8, 128), (32, 4, 64)])
@pytest.mark.parametrize("lengths", [MIDDLE, SHORTER])
def test_prefill_two_groups_per_tile(device, hq, hkv, dh, lengths) -> None:
    _check(device, torch.bfloat16, hq, hkv, dh, lengths)
    order = torch.tensor([3, 0, 4, 1, 2], dtype=torch.int32, device=device)
    _check(device, torch.float16, hq, hkv, dh, lengths, seq_order=order)


# 32 / 8 heads at Dh 128, around one and two rounds of two-group workgroups: one sequence on each
# side of the rules by its mean keys, ragged chunks over more than one round, and chunks that
# stay with one group for their keys or their number.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lengths", [
    ([569], [569]), ([1051], [569]), ([1972], [569]), ([1323], [1323]), ([2100], [1323]),
    ([3267, 1419, 556, 1209, 1969], [233, 385, 198, 88, 254]),
    ([1700, 1650, 1601, 1500, 1, 1690], [266, 257, 289, 290, 1, 260]),
    ([2100, 2050, 400], [700, 700, 400])])
def test_prefill_forms(device, dtype, lengths) -> None:
    _check(device, dtype, 32, 8, 128, lengths)
