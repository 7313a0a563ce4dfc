// The MFMA decode (decode_pv.hpp) over blocks of 16 tokens, and its dispatch.
#include "decode_pv.hpp"

namespace tks {

bool decode_mfma_supported(int32_t dtype, int32_t head_dim, int32_t group, int32_t block_size,
                           int64_t num_blocks, int32_t num_kv_heads) {
  if (dtype != TKS_BFLOAT16 && dtype != TKS_FLOAT16) return false;
  if (block_size % 16 != 0) return false;
  // Page ids (16 rows of one head) of the layer are 32-bit.
  if (num_blocks * num_kv_heads * (block_size / 16) >= (int64_t{1} << 31)) return false;
  if (head_dim == 128) return group == 1 || group == 2 || group == 4 || group == 8;
  if (head_dim == 64) return group == 2 || group == 4 || group == 8 || group == 16;
  return false;
}

int32_t launch_decode_mfma(const DecodeArgs &a, int32_t dtype, int32_t num_seqs,
                           int32_t num_kv_heads, int32_t group, int32_t head_dim,
                           hipStream_t stream, bool fp8_pools) {
  return a.block_pages == 1 ? launch_pv<false>(a, dtype, num_seqs, num_kv_heads, group, head_dim,
                                               stream, fp8_pools)
                            : launch_decode_blocks(a, dtype, num_seqs, num_kv_heads, group,
                                                   head_dim, stream, fp8_pools);
}

}  // namespace tks
