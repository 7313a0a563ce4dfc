"""16-bit decode over e4m3 pools with the library's own, longer key splits (256 to 1,023
(sequence, KV head) pairs and a bound of 4,096 keys or more) against the fp32 oracle:
lengths around the 1,280-key splits and blocks that do not divide them.

Tolerance: the result's one rounding to bf16 (2^-8 relative) and 2e-5 absolute for fp32 sums
in another order, plus the probabilities' rounding to bf16 in P.V over blocks of 16 (2^-9
relative of each product; at most 2^-9 times the largest |v|, under 2e-2).
"""

import pytest
import torch
from torch.testing import assert_close

from oracle import paged
from tokserve_amd import workloads
from tokserve_amd.kernels import ops

pytestmark = pytest.mark.gpu

CONTEXTS = [4100, 1279, 1280, 1281, 2560, 2561, 1, 0] + [17 + 61 * i for i in range(56)]


@pytest.mark.parametrize("granularity", ["pool", "row"])
@pytest.mark.parametrize("block_size", [16, 48])
def test_fp8_decode_splits(device, granularity, block_size) -> None:
    kw = (dict(scale_granularity="row") if granularity == "row"
          else dict(k_scale=0.5, v_scale=0.25))
    batch = workloads.paged_batch(CONTEXTS, [1] * len(CONTEXTS), num_q_heads=8, num_kv_heads=4,
                                  head_dim=64, block_size=block_size, dtype=torch.bfloat16,
                                  device=device, seed=2, kv_dtype=torch.float8_e4m3fn, **kw)
    out = ops.paged_attention_decode(
        batch.query, batch.key_cache, batch.value_cache, batch.block_tables, batch.seq_lens,
        layer_index=0, max_seq_len=batch.max_seq_len, **batch.scale_kwargs)
    torch.cuda.synchronize()
    pools = []
    for cache, scale, scales in ((batch.key_cache, batch.k_scale, batch.k_scales),
                                 (batch.value_cache, batch.v_scale, batch.v_scales)):
        pool = cache.cpu().float()
        pools.append(pool * (scale if scales is None else scales.cpu().unsqueeze(-1)))
    expected = paged.decode_batch(batch.query.cpu().float(), *pools, batch.block_tables.cpu(),
                                  batch.seq_lens.cpu(), 0, torch.float32)
    assert_close(out.cpu().float(), expected, rtol=2.0 ** -8, atol=2e-2)
