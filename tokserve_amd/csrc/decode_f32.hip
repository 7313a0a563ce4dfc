// Paged decode for fp32 queries, both products in fp32 on the matrix cores
// (v_mfma_f32_16x16x4_f32), over fp32 or e4m3 pools whose block size is a multiple of 16.
//
// Bound: HBM for large batches, the chain of dependent reads for small ones. One workgroup
// of W waves per (sequence, KV head[, key split]); the waves take contiguous ranges of
// 16-key pages and merge their softmax states through LDS at the end. The G query heads are
// the (up to 16) columns of one MFMA tile. K and V go from memory straight into the MFMA
// operands, no LDS between: one MFMA contracts any four values of which lane (g, r) holds
// the g-th, so a lane takes consecutive ones and reads 16 bytes at a time:
//   S (16 keys x 16 heads) = K . Q^T: lane (g, r) holds parts of key r's row;
//   O^T (dims x 16 heads) += V^T . P^T: MFMA i contracts keys 4 g + i, the keys whose
//     probabilities lane (g, r) already holds, over the dims lane r read of them.
// The next page's loads are in flight while a page is used (16 KB per wave at Dh 128).
// Against the VALU kernel: 128 sequences of up to 8,192 keys (32 / 8 heads, Dh 128) 1,214
// -> 387 us (5.1 TB/s), 128 of up to 1,152 (32 / 4, Dh 64, RoPE and append included) 93 ->
// 38 us, 33 over e4m3 pools with row scales 730 -> 60 us, the small step (8 sequences of up
// to 513 keys, 8 / 2, Dh 64, three launches before) 27 -> 12.6 us.
//
// ROPE: RoPE and the KV append of the new tokens in the same launch, as in decode_pv.hpp:
// the query is rotated while it is staged, and the wave with the sequence's last page
// rotates the new key row, uses both new rows in place of what the pool holds in their
// slot, and writes them there.
#include "attention_common.hpp"
#include "rope_common.hpp"

namespace tks {
namespace {

constexpr int kFPage = 16;

// A lane's share of a page. K: key r's dims k_dim(0 .. DH / 4 - 1, g); V: keys 4 g + i,
// dims v_dim(0 .. DH / 16 - 1, r) of each.
template <typename KV, int DH>
struct LanePage;
template <int DH>
struct LanePage<float, DH> {
  static constexpr int KN = DH / 16, VN = DH / 64;
  uint4 k[KN], v[4][VN];
  static __device__ __forceinline__ int k_dim(int x, int g) { return 16 * (x / 4) + 4 * g + x % 4; }
  static __device__ __forceinline__ int v_dim(int d, int m) { return 64 * (d / 4) + 4 * m + d % 4; }
  __device__ __forceinline__ void load(const float *kp, const float *vp, int g, int r) {
#pragma unroll
    for (int j = 0; j < KN; ++j) k[j] = ld16_stream(kp + r * DH + 16 * j + 4 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int h = 0; h < VN; ++h) v[i][h] = ld16_stream(vp + (4 * g + i) * DH + 64 * h + 4 * r);
  }
  // Row `row` of the page from LDS instead.
  __device__ __forceinline__ void take_row(int row, const float *k_s, const float *v_s, int g,
                                           int r) {
    if (r == row) {
#pragma unroll
      for (int j = 0; j < KN; ++j) k[j] = ld16(k_s + 16 * j + 4 * g);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (4 * g + i == row) {
#pragma unroll
        for (int h = 0; h < VN; ++h) v[i][h] = ld16(v_s + 64 * h + 4 * r);
      }
  }
  __device__ __forceinline__ void k_row(float *x) const {
#pragma unroll
    for (int j = 0; j < KN; ++j) unpack<float>(k[j], x + 4 * j);
  }
  __device__ __forceinline__ void v_row(int i, float *x) const {
#pragma unroll
    for (int h = 0; h < VN; ++h) unpack<float>(v[i][h], x + 4 * h);
  }
};
template <int DH>
struct LanePage<fp8e4m3_t, DH> {
  static constexpr int KN = DH / 64, VN = DH / 64;
  uint4 k[KN];
  uint32_t v[4][VN];
  static __device__ __forceinline__ int k_dim(int x, int g) { return 64 * (x / 16) + 16 * g + x % 16; }
  static __device__ __forceinline__ int v_dim(int d, int m) { return DH / 16 * m + d; }
  __device__ __forceinline__ void load(const fp8e4m3_t *kp, const fp8e4m3_t *vp, int g, int r) {
#pragma unroll
    for (int j = 0; j < KN; ++j) k[j] = ld16_stream(kp + r * DH + 64 * j + 16 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t *p = reinterpret_cast<const uint32_t *>(vp + (4 * g + i) * DH + DH / 16 * r);
#pragma unroll
      for (int h = 0; h < VN; ++h) v[i][h] = __builtin_nontemporal_load(p + h);
    }
  }
  __device__ __forceinline__ void k_row(float *x) const {
#pragma unroll
    for (int j = 0; j < KN; ++j) unpack<fp8e4m3_t>(k[j], x + 16 * j);
  }
  __device__ __forceinline__ void v_row(int i, float *x) const {
#pragma unroll
    for (int h = 0; h < VN; ++h) fp8x4_to_float(v[i][h], x + 4 * h);
  }
};

template <int N>
struct PageSlot {
  static constexpr int value = N;
};

// The new token's key row (rotated at its position) and value row into k_s and v_s, by one
// wave; whether slot a.slots[b] lies in the pool (a negative slot appends nothing).
template <int DH>
__device__ __forceinline__ bool stage_rows(const DecodeArgs &a, int b, int kvh, int lane,
                                           float *k_s, float *v_s) {
  constexpr int HALF = DH / 2;
  const int64_t slot = a.slots[b];
  if (slot < 0 || slot >= a.pool.num_blocks * a.pool.block_size) return false;
  if (lane < HALF / 4) {
    const float *kn = static_cast<const float *>(a.k_new) + b * a.kn_ss + (int64_t)kvh * a.kn_hs;
    const int64_t pos = min(max(a.positions[b], (int64_t)0), a.table_len - 1);
    float cf[4], sf[4], o1[4], o2[4];
    load_table<float, 4>(static_cast<const float *>(a.cos_t) + pos * HALF,
                         static_cast<const float *>(a.sin_t) + pos * HALF, lane * 4, cf, sf);
    rotate_values<float, 4>(kn + lane * 4, cf, sf, HALF, o1, o2);
    store_pair<float, 4>(k_s + lane * 4, o1, o2, HALF);
  } else if (lane >= 32 && lane < 32 + DH / 4) {
    const float *vn = static_cast<const float *>(a.v_new) + b * a.vn_ss + (int64_t)kvh * a.vn_hs;
    st16(v_s + (lane - 32) * 4, ld16(vn + (lane - 32) * 4));
  }
  return true;
}

// The staged rows into the pool.
template <int DH>
__device__ __forceinline__ void write_rows(const DecodeArgs &a, int b, int kvh, int lane,
                                           const float *k_s, const float *v_s) {
  const int64_t slot = a.slots[b];
  const int64_t blk = slot / a.pool.block_size;
  const int64_t row = a.pool.layer_base + blk * a.pool.block_stride +
                      (int64_t)kvh * a.pool.head_stride + (slot - blk * a.pool.block_size) * DH;
  float *kd = static_cast<float *>(const_cast<void *>(a.kc)) + row;
  float *vd = static_cast<float *>(const_cast<void *>(a.vc)) + row;
  if (lane < DH / 4) {
    st16(kd + lane * 4, ld16(k_s + lane * 4));
    st16(vd + lane * 4, ld16(v_s + lane * 4));
  }
}

// Orders a wave's own LDS writes and reads.
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename KV, int DH, int W, bool ROPE, bool ROWS>
__global__ __launch_bounds__(64 * W) void decode_f32_kernel(DecodeArgs a, int G) {
  typedef LanePage<KV, DH> Page;
  constexpr int KD = DH / 4, VD = DH / 16;
  static_assert(!ROPE || sizeof(KV) == 4, "fused append: fp32 pools");
  __shared__ __attribute__((aligned(16))) float q_s[16 * DH];
  __shared__ __attribute__((aligned(16))) float acc_s[W][16][DH];
  __shared__ float m_s[W][16], l_s[W][16];
  __shared__ __attribute__((aligned(16))) float nk_s[ROPE ? DH : 4], nv_s[ROPE ? DH : 4];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int kvh = blockIdx.x, split = blockIdx.z;
  const int b = a.seq_order ? min(max(a.seq_order[blockIdx.y], 0), (int)gridDim.y - 1)
                            : (int)blockIdx.y;
  const int seq_len = a.seq_lens[b];
  const int len = min(seq_len, a.key_cap);
  const int n_pages = (len + kFPage - 1) / kFPage;
  const int p_begin = split * a.pages_per_split;
  float *out = static_cast<float *>(a.out) + b * a.o_ss + (int64_t)kvh * G * a.o_hs;
  if (p_begin >= n_pages) {
    if (split == 0) {  // no keys: a zero row (and the new rows are appended all the same)
      for (int i = threadIdx.x; i < G * DH; i += 64 * W)
        out[(int64_t)(i / DH) * a.o_hs + i % DH] = 0.f;
      if constexpr (ROPE) {
        if (n_pages == 0 && wave == 0 && stage_rows<DH>(a, b, kvh, lane, nk_s, nv_s)) {
          lds_order();
          write_rows<DH>(a, b, kvh, lane, nk_s, nv_s);
        }
      }
    }
    return;
  }
  const int p_end = min(n_pages, p_begin + a.pages_per_split);
  const int per_wave = (p_end - p_begin + W - 1) / W;
  const int w_begin = min(p_end, p_begin + wave * per_wave);
  const int w_end = min(p_end, w_begin + per_wave);

  const int64_t head_base = a.pool.layer_base + (int64_t)kvh * a.pool.head_stride;
  const KV *kc = static_cast<const KV *>(a.kc) + head_base;
  const KV *vc = static_cast<const KV *>(a.vc) + head_base;
  const int32_t *bt_row = a.bt + (int64_t)b * a.bt_stride;
  const int block_pages = a.block_pages;
  const int page_stride = block_pages * (int)gridDim.x;  // pages of this layer per block

  // Lane i: the id of page c0 + i, in pages of 16 rows behind this head's first.
  auto page_ids = [&](int c0) {
    if (c0 + lane >= w_end) return 0;
    const int at = block_pages == 1 ? c0 + lane : (c0 + lane) / block_pages;
    return (int)block_of(bt_row, at, a.pool.num_blocks) * page_stride + (c0 + lane) -
           at * block_pages;
  };
  Page pages[2];
  float ks4[2][4], vs4[2][4];  // ROWS: the lane's keys' scales
  auto load = [&](auto slot_c, int ids, int idx) {
    constexpr int S = decltype(slot_c)::value;
    const int64_t row = (int64_t)__builtin_amdgcn_readlane(ids, idx) * kFPage;
    pages[S].load(kc + row * DH, vc + row * DH, g, r);
    if constexpr (ROWS) {
      const int64_t at = head_base / DH + row + 4 * g;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ks4[S][i] = a.k_rs[at + i];
        vs4[S][i] = a.v_rs[at + i];
      }
    }
  };
  int ids = page_ids(w_begin);
  const bool some = w_begin < w_end;
  if (some) load(PageSlot<0>{}, ids, 0);

  // The query rows through LDS, rotated there with ROPE.
  bool staged = false, patch = false;
  if constexpr (ROPE) {
    if (some && w_end == n_pages) {  // wave-uniform
      staged = stage_rows<DH>(a, b, kvh, lane, nk_s, nv_s);
      patch = staged && seq_len == len;
      lds_order();
    }
  }
  {
    const float *q = static_cast<const float *>(a.q) + b * a.q_ss + (int64_t)kvh * G * a.q_hs;
    if constexpr (ROPE) {
      constexpr int HALF = DH / 2;
      for (int t = threadIdx.x; t < G * HALF / 4; t += 64 * W) {
        const int64_t pos = min(max(a.positions[b], (int64_t)0), a.table_len - 1);
        const int h = t / (HALF / 4), j = (t % (HALF / 4)) * 4;
        float cf[4], sf[4], o1[4], o2[4];
        load_table<float, 4>(static_cast<const float *>(a.cos_t) + pos * HALF,
                             static_cast<const float *>(a.sin_t) + pos * HALF, j, cf, sf);
        rotate_values<float, 4>(q + (int64_t)h * a.q_hs + j, cf, sf, HALF, o1, o2);
        store_pair<float, 4>(&q_s[h * DH + j], o1, o2, HALF);
      }
    } else {
      for (int t = threadIdx.x; t < G * DH / 4; t += 64 * W) {
        const int h = t / (DH / 4), j = (t % (DH / 4)) * 4;
        st16(&q_s[h * DH + j], ld16(q + (int64_t)h * a.q_hs + j));
      }
    }
  }
  __syncthreads();
  float qf[KD];  // head column r (columns past G repeat the last: computed, not used)
  {
    const float *row = &q_s[min(r, G - 1) * DH];
#pragma unroll
    for (int x = 0; x < KD; ++x) qf[x] = row[Page::k_dim(x, g)];
  }

  f32x4 acc[VD];
#pragma unroll
  for (int d = 0; d < VD; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Softmax of head column r in log2 units: m the reference (it moves when a score passes
  // it by more than 8), l this lane's share of the sum.
  float m = -INFINITY, l = 0.f;
  const float scale_log2 = a.scale_log2;
  const int new_off = ROPE ? (len - 1) % kFPage : 0;

  auto consume = [&](auto slot_c, int p) {
    constexpr int S = decltype(slot_c)::value;
    const bool last = p == n_pages - 1;
    if constexpr (ROPE) {
      if (patch && last) pages[S].take_row(new_off, nk_s, nv_s, g, r);
    }
    float k[KD];
    pages[S].k_row(k);
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < KD; ++x) s = mfma_f32(k[x], qf[x], s);
    if constexpr (ROWS) {
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] *= ks4[S][i];
    }
    float sv[4];
    bool valid[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      valid[i] = !last || p * kFPage + 4 * g + i < len;
      sv[i] = valid[i] ? s[i] * scale_log2 : -INFINITY;
    }
    const float top = nan_max(nan_max(sv[0], sv[1]), nan_max(sv[2], sv[3]));
    if (__builtin_amdgcn_ballot_w64(top > m + 8.f)) {
      const float mx = xgroup_max(top);
      const bool bump = mx > m + 8.f;
      const float alpha = bump ? fast_exp2(m - mx) : 1.f;
      m = bump ? mx : m;
      l *= alpha;
#pragma unroll
      for (int d = 0; d < VD; ++d) acc[d] *= alpha;
    }
    const float nr = m == -INFINITY ? 0.f : -m;
    float pv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      pv[i] = valid[i] ? fast_exp2(__builtin_fmaf(s[i], scale_log2, nr)) : 0.f;
    l += (pv[0] + pv[1]) + (pv[2] + pv[3]);
    if constexpr (ROWS) {
#pragma unroll
      for (int i = 0; i < 4; ++i) pv[i] = valid[i] ? pv[i] * vs4[S][i] : 0.f;
    }
    // A page's sums start from zero and are then added: shorter chains of roundings.
    f32x4 o[VD] = {};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v[VD];
      pages[S].v_row(i, v);
#pragma unroll
      for (int d = 0; d < VD; ++d)  // past the last key the pool holds anything: 0 * NaN
        o[d] = mfma_f32(valid[i] ? v[d] : 0.f, pv[i], o[d]);
    }
#pragma unroll
    for (int d = 0; d < VD; ++d) acc[d] += o[d];
  };

  // Loads past the range repeat its last page (an unconditional load keeps the compiler
  // from waiting for the one in flight).
  for (int c0 = w_begin; c0 < w_end; c0 += 64) {
    const int n = min(w_end - c0, 64);
    if (c0 != w_begin) {
      ids = page_ids(c0);
      load(PageSlot<0>{}, ids, 0);
    }
    for (int i = 0; i < n; i += 2) {
      load(PageSlot<1>{}, ids, min(i + 1, n - 1));
      consume(PageSlot<0>{}, c0 + i);
      if (i + 1 >= n) break;
      load(PageSlot<0>{}, ids, min(i + 2, n - 1));
      consume(PageSlot<1>{}, c0 + i + 1);
    }
  }
  if constexpr (ROPE) {
    if (staged) write_rows<DH>(a, b, kvh, lane, nk_s, nv_s);  // this wave has read its page
  }

  l = xgroup_sum(l);
  if (r < G) {
    if (g == 0) {
      m_s[wave][r] = m;
      l_s[wave][r] = l;
    }
#pragma unroll
    for (int d = 0; d < VD; ++d)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc_s[wave][r][Page::v_dim(d, 4 * g + i)] = acc[d][i];
  }
  __syncthreads();
  for (int x = threadIdx.x; x < G * DH; x += 64 * W) {
    const int h = x / DH, d = x % DH;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; ++w) M = fmaxf(M, m_s[w][h]);
    float L = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float e = m_s[w][h] == -INFINITY ? 0.f : fast_exp2(m_s[w][h] - M);
      L += e * l_s[w][h];
      o += e * acc_s[w][h][d];
    }
    if (a.max_splits == 1) {
      out[(int64_t)h * a.o_hs + d] = o / L * a.v_scale;
    } else {
      const int64_t w = ((int64_t)b * a.num_q_heads + kvh * G + h) * a.max_splits + split;
      if (d == 0) {
        a.ws_m[w] = M;
        a.ws_l[w] = L;
      }
      a.ws_acc[w * DH + d] = o * a.v_scale;
    }
  }
}

template <typename KV, int DH, int W>
int32_t launch_waves(const DecodeArgs &a, int G, dim3 grid, hipStream_t s) {
  if constexpr (sizeof(KV) == 4) {
    if (a.positions != nullptr)
      decode_f32_kernel<KV, DH, W, true, false><<<grid, 64 * W, 0, s>>>(a, G);
    else
      decode_f32_kernel<KV, DH, W, false, false><<<grid, 64 * W, 0, s>>>(a, G);
  } else if (a.k_rs != nullptr) {
    decode_f32_kernel<KV, DH, W, false, true><<<grid, 64 * W, 0, s>>>(a, G);
  } else {
    decode_f32_kernel<KV, DH, W, false, false><<<grid, 64 * W, 0, s>>>(a, G);
  }
  return check_launch();
}

template <typename KV>
int32_t launch_kv(const DecodeArgs &a, int G, int32_t head_dim, bool wide, dim3 grid,
                  hipStream_t s) {
  if (head_dim == 64)
    return wide ? launch_waves<KV, 64, 8>(a, G, grid, s) : launch_waves<KV, 64, 4>(a, G, grid, s);
  return wide ? launch_waves<KV, 128, 8>(a, G, grid, s) : launch_waves<KV, 128, 4>(a, G, grid, s);
}

}  // namespace

bool decode_f32_supported(int32_t head_dim, int32_t group, int32_t block_size, int64_t num_blocks,
                          int32_t num_kv_heads) {
  return (head_dim == 64 || head_dim == 128) && group >= 1 && group <= 16 &&
         block_size % 16 == 0 &&
         num_blocks * num_kv_heads * (block_size / 16) < (int64_t{1} << 31);
}

int32_t launch_decode_f32(const DecodeArgs &a, int32_t num_seqs, int32_t num_kv_heads,
                          int32_t group, int32_t head_dim, bool wide, bool fp8_pools,
                          hipStream_t stream) {
  const dim3 grid(num_kv_heads, num_seqs, a.max_splits);
  return fp8_pools ? launch_kv<fp8e4m3_t>(a, group, head_dim, wide, grid, stream)
                   : launch_kv<float>(a, group, head_dim, wide, grid, stream);
}

}  // namespace tks
