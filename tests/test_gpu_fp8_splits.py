"""16-bit decode over e4m3 pools with the library's own key splits (256 to 1,023 (sequence, KV
head) pairs and a bound of 4,096 keys or more) against the fp32 oracle: lengths around the
splits, of 1,280 keys or, for fewer pairs at Dh 64, 512, and blocks that do not divide them.

The keys at the ends of splits, pages and sequences have values of 64 among N(0, 1) ones: one of
them left out or taken twice moves a result by about 64 / 4,100 or more, several tolerances.

Tolerance, for each element: the probabilities' rounding to bf16 in P.V over blocks of 16 (2^-9
relative of each product, at most 2^-9 times the sum of p |v|), the result's one rounding to
bf16 (2^-8 relative) and 2e-5 for fp32 sums in another order.
"""

import pytest
import torch

from oracle import paged
from tokserve_amd import workloads
from tokserve_amd.kernels import ops

pytestmark = pytest.mark.gpu

CONTEXTS = [4100, 1279, 1280, 1281, 2560, 2561, 1, 0] + [17 + 61 * i for i in range(56)]
SPLITS = {4: 512, 8: 1280}  # KV heads of the 64 sequences: keys per split
LARGE = 64.0


def _mark(batch, block_size: int, split: int) -> None:
    """Values of +-LARGE (by dim) at the first and last keys of splits and sequences."""

    tables = batch.block_tables.cpu()
    for b, n in enumerate(batch.contexts):
        ends = {p for e in range(0, n, split) for p in (e - 16, e - 1, e, e + 15)} | {n - 1}
        for p in sorted(p for p in ends if 0 <= p < n):
            block, row = int(tables[b, p // block_size]), p % block_size
            sign = torch.where(torch.arange(batch.value_cache.shape[4]) % 3 == p % 3, -1.0, 1.0)
            if batch.v_scales is None:
                code = sign * (LARGE / batch.v_scale)
            else:
                code = sign * 448.0
                batch.v_scales[0, block, :, row] = LARGE / 448.0
            batch.value_cache[0, block, :, row] = code.to(batch.value_cache.dtype).to(
                batch.value_cache.device)


@pytest.mark.parametrize("granularity", ["pool", "row"])
@pytest.mark.parametrize("block_size", [16, 48])
@pytest.mark.parametrize("kv_heads", [4, 8])
def test_fp8_decode_splits(device, granularity, block_size, kv_heads) -> None:
    kw = (dict(scale_granularity="row") if granularity == "row"
          else dict(k_scale=0.5, v_scale=0.25))
    batch = workloads.paged_batch(CONTEXTS, [1] * len(CONTEXTS), num_q_heads=2 * kv_heads,
                                  num_kv_heads=kv_heads, head_dim=64, block_size=block_size,
                                  dtype=torch.bfloat16, device=device, seed=2,
                                  kv_dtype=torch.float8_e4m3fn, **kw)
    _mark(batch, block_size, SPLITS[kv_heads])
    out = ops.paged_attention_decode(
        batch.query, batch.key_cache, batch.value_cache, batch.block_tables, batch.seq_lens,
        layer_index=0, max_seq_len=batch.max_seq_len, **batch.scale_kwargs)
    torch.cuda.synchronize()
    pools = []
    for cache, scale, scales in ((batch.key_cache, batch.k_scale, batch.k_scales),
                                 (batch.value_cache, batch.v_scale, batch.v_scales)):
        pool = cache.cpu().float()
        pools.append(pool * (scale if scales is None else scales.cpu().unsqueeze(-1)))

    def oracle(values):
        return paged.decode_batch(batch.query.cpu().float(), pools[0], values,
                                  batch.block_tables.cpu(), batch.seq_lens.cpu(), 0,
                                  torch.float32)

    expected = oracle(pools[1])
    bound = 2.0 ** -9 * oracle(pools[1].abs()) + 2.0 ** -8 * expected.abs() + 2e-5
    worst = ((out.cpu().float() - expected).abs() / bound).max()
    assert worst <= 1.0, f"{worst:.2f} times the tolerance"
