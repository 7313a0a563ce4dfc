"""The decode's key splits by block size, read off the workspace sizes (CPU)."""

import pytest

from tokserve_amd.kernels import ops


@pytest.mark.parametrize("block_size", [32, 48, 64, 256])
@pytest.mark.parametrize("seqs", [1, 5, 31, 32, 100, 127, 128])
@pytest.mark.parametrize("blocks_of_768", [1, 4, 5, 6, 11, 40])
def test_long_blocks_split_as_blocks_of_16(block_size, seqs, blocks_of_768) -> None:
    """Blocks that are multiples of 16 get the splits of blocks of 16, rounded up to whole
    blocks: never more partials, and as many where 256 keys are whole blocks."""

    def partials(bs):
        return ops.decode_workspace_bytes(seqs, 32, 8, 128, bs, 768 * blocks_of_768, 0)

    assert partials(block_size) <= partials(16)
    if 256 % block_size == 0 and (seqs == 31 or seqs >= 32):  # splits of 768 or 512 keys, or none
        assert partials(block_size) == partials(16)


@pytest.mark.parametrize("block_size", [1, 2, 8, 24])
def test_other_blocks_keep_their_block_counts(block_size) -> None:
    """16 to 48 blocks to a split for a batch too small to fill the GPU, 32 for a middling
    one of long sequences."""

    few = ops.decode_workspace_bytes(8, 32, 8, 128, block_size, 1000 * block_size, 0)
    assert few == ops.decode_workspace_bytes(8, 32, 8, 128, block_size, 1000 * block_size, 48)
    mid = ops.decode_workspace_bytes(64, 32, 8, 128, block_size, 1000 * block_size, 0)
    assert mid == ops.decode_workspace_bytes(64, 32, 8, 128, block_size, 1000 * block_size, 32)
