"""The operators' native device kernels: errors as _lib.check raises them, and scratch memory
that belongs to one call."""

import pytest
import torch

from tokserve_amd import workloads
from tokserve_amd.kernels import ops, torch_ops

pytestmark = pytest.mark.gpu

_ops = torch.ops.tokserve_amd


def test_native_kernels_raise_the_reference_exceptions(device) -> None:
    assert torch_ops.NATIVE_LIBRARY.is_file()
    batch = workloads.paged_batch([20], [1], num_q_heads=4, num_kv_heads=2, head_dim=64,
                                  block_size=16, dtype=torch.bfloat16, device=device, seed=0)
    with pytest.raises(IndexError, match="paged_attention_decode: layer_index is out of range"):
        ops.paged_attention_decode(batch.query, batch.key_cache, batch.value_cache,
                                   batch.block_tables, batch.seq_lens, layer_index=1,
                                   max_seq_len=20)
    x = torch.zeros(2, 8, dtype=torch.int32, device=device)
    with pytest.raises(TypeError, match="unsupported dtype torch.int32"):
        _ops.greedy_argmax(x, torch.empty(2, 1, dtype=torch.int64, device=device))
    small = torch.empty(8, dtype=torch.uint8, device=device)
    with pytest.raises(ValueError):
        ops.paged_attention_decode(batch.query, batch.key_cache, batch.value_cache,
                                   batch.block_tables, batch.seq_lens, layer_index=0,
                                   max_seq_len=20, pages_per_split=1, workspace=small)


def test_split_decodes_on_two_streams_keep_their_partials_apart(device) -> None:
    batches = [workloads.paged_batch([700 + 100 * i, 90, 1300], [1] * 3, num_q_heads=8,
                                     num_kv_heads=2, head_dim=128, block_size=16,
                                     dtype=torch.bfloat16, device=device, seed=i)
               for i in range(2)]

    def decode(batch):
        return ops.paged_attention_decode(batch.query, batch.key_cache, batch.value_cache,
                                          batch.block_tables, batch.seq_lens, layer_index=0,
                                          max_seq_len=batch.max_seq_len, pages_per_split=4)

    expected = [decode(batch) for batch in batches]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in batches]
    outs: list = [[], []]
    for _ in range(20):
        for i, batch in enumerate(batches):
            with torch.cuda.stream(streams[i]):
                outs[i].append(decode(batch))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(out, expected[i]) for out in outs[i])


@pytest.mark.parametrize("granularity", ["pool", "row"])
def test_fp8_prefills_on_two_streams_keep_their_pages_apart(device, granularity) -> None:
    """The decoded pages of a call are its own: nothing per device is kept for them, and calls
    on two streams give what they give alone."""

    kw = (dict(scale_granularity="row") if granularity == "row"
          else dict(k_scale=0.5, v_scale=0.25))
    batches = [workloads.paged_batch([2000 + 300 * i, 90, 1300], [40, 90, 300], num_q_heads=32,
                                     num_kv_heads=8, head_dim=128, block_size=16,
                                     dtype=torch.bfloat16, device=device, seed=i,
                                     kv_dtype=torch.float8_e4m3fn, **kw)
               for i in range(2)]

    def prefill(batch):
        return ops.paged_attention_prefill(batch.query, batch.key_cache, batch.value_cache,
                                           batch.block_tables, batch.seq_lens,
                                           batch.cu_seqlens_q, layer_index=0,
                                           max_query_len=batch.max_query_len,
                                           max_seq_len=batch.max_seq_len, **batch.scale_kwargs)

    kept = dict(torch_ops._workspaces)
    expected = [prefill(batch) for batch in batches]
    assert torch_ops._workspaces == kept
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in batches]
    outs: list = [[], []]
    for _ in range(10):
        for i, batch in enumerate(batches):
            with torch.cuda.stream(streams[i]):
                outs[i].append(prefill(batch))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(out, expected[i]) for out in outs[i])
