// The MFMA decode (decode_pv.hpp) over blocks of several 16-token pages.
#include "decode_pv.hpp"

namespace tks {

int32_t launch_decode_blocks(const DecodeArgs &a, int32_t dtype, int32_t num_seqs,
                             int32_t num_kv_heads, int32_t group, int32_t head_dim,
                             hipStream_t stream, bool fp8_pools) {
  return launch_pv<true>(a, dtype, num_seqs, num_kv_heads, group, head_dim, stream, fp8_pools);
}

}  // namespace tks
