// Chunked-prefill paged attention for fp32 queries, both products in fp32 on the matrix
// cores (v_mfma_f32_16x16x4_f32), over fp32 or e4m3 pools of any block size.
//
// Bound: the fp32 MFMA rate, 256 flop per CU and cycle (157 TFLOP/s at 2.4 GHz, a 16th of
// bf16's), and the VALU beside it (one does not hide the other: a step's 64 MFMAs take
// 2,048 cycles of a SIMD, its about 130 VALU instructions some 600). 16 prompts of 64 to
// 1,024 tokens (32 / 4 heads, Dh 64): 828 us on the VALU kernel, 117 us here (92 TFLOP/s
// of visible scores). One workgroup of 4 waves per (sequence, KV head, 64 rows), row =
// query token * G + query head, 16 rows a wave. Two 16-row tiles a wave halve the loads
// but also the workgroups, and the longest of them then set the time: 152 us.
//
// Operands. One MFMA contracts four values, lane (g, r) holding A[r][g] and B[g][r], and
// yields D[4 g + i][r]. Which four is free as long as A and B agree, so both products pick
// the ones that make LDS reads 16 bytes wide and keep the probabilities in their lanes:
//   S^T (16 keys x 16 rows) = K . Q^T: MFMA (j, e) contracts dims 16 j + 4 g + e, so lane
//     (g, r) reads key r's dims 16 j + 4 g .. +3 at once;
//   O^T (16 dims x 16 rows) += V^T . P^T: MFMA i contracts keys 4 g + i, the keys whose
//     scores lane (g, r) holds in S^T; A's row m of dim tile d is dim 4 m + d (of each 64),
//     so lane (g, r) reads key 4 g + i's dims 4 r .. +3 at once for four dim tiles.
// K and V go through registers into a double-buffered LDS tile of 32 keys (e4m3 codes are
// decoded on the way; per-row scales stay beside the tile and multiply scores and
// probabilities). Rows are padded by 16 bytes against bank conflicts.
#include "attention_common.hpp"

#include <algorithm>

namespace tks {
namespace {

constexpr int kFWaves = 4;
constexpr int kFKeys = 32;  // keys per step
constexpr int kFRows = kFWaves * 16;

// This thread's part of one K (or V) row of a step, as loaded: DH / 8 elements.
template <typename KV, int DH>
struct RowPart;
template <int DH>
struct RowPart<float, DH> {
  static constexpr int N = DH / 32;  // 16-byte chunks c, c + 8, ... of the row
  uint4 v[N];
  __device__ __forceinline__ void load(const float *row, int c) {
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = ld16(row + (c + 8 * j) * 4);
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = make_uint4(0, 0, 0, 0);
  }
  __device__ __forceinline__ void store(float *row, int c) const {
#pragma unroll
    for (int j = 0; j < N; ++j) st16(row + (c + 8 * j) * 4, v[j]);
  }
};
template <int DH>
struct RowPart<fp8e4m3_t, DH> {
  static constexpr int N = DH / 32;  // words: codes 4 N c .. of the row
  uint32_t w[N];
  __device__ __forceinline__ void load(const fp8e4m3_t *row, int c) {
    if constexpr (N == 4) {
      const uint4 u = ld16(row + 16 * c);
      w[0] = u.x, w[1] = u.y, w[2] = u.z, w[3] = u.w;
    } else {
      const uint2 u = *reinterpret_cast<const uint2 *>(row + 8 * c);
      w[0] = u.x, w[1] = u.y;
    }
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int j = 0; j < N; ++j) w[j] = 0;
  }
  __device__ __forceinline__ void store(float *row, int c) const {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      float f[4];
      fp8x4_to_float(w[j], f);
      *reinterpret_cast<float4 *>(row + 4 * (N * c + j)) = make_float4(f[0], f[1], f[2], f[3]);
    }
  }
};

// Dh 128: nothing is scheduled across this point, which keeps the operands of one 64-dim
// group at a time in registers.
template <int DH>
__device__ __forceinline__ void register_fence() {
#if __HIP_DEVICE_COMPILE__
  if constexpr (DH == 128) __builtin_amdgcn_sched_barrier(0);
#endif
}

template <int N>
struct Slot {
  static constexpr int value = N;
};

// One query row on the VALU, by one wave: lane t scores key k0 + t of each 64, then
// accumulates dims t (and t + 64).
template <typename KV, int DH>
__device__ __forceinline__ void one_row(const PrefillArgs &a, int qh, const KV *kc, const KV *vc,
                                        int64_t head_base, const int32_t *bt_row, int token,
                                        int n_keys, int lane) {
  const uint32_t BS = a.pool.block_size;
  const float *q = static_cast<const float *>(a.q) + (int64_t)token * a.q_ts + (int64_t)qh * a.q_hs;
  float m = -INFINITY, l = 0.f, acc[DH / 64] = {};
#pragma unroll 1
  for (int k0 = 0; k0 < n_keys; k0 += 64) {
    const uint32_t key = min(k0 + lane, n_keys - 1);
    const int64_t at = block_of(bt_row, key / BS, a.pool.num_blocks) * a.pool.block_stride +
                       (int64_t)(key % BS) * DH;
    float s = 0.f;
#pragma unroll 1
    for (int d = 0; d < DH; ++d) s += q[d] * to_float(kc[at + d]);
    s *= a.scale_log2;
    float vs = 1.f;
    if (a.k_rs != nullptr) {
      s *= a.k_rs[(head_base + at) / DH];
      vs = a.v_rs[(head_base + at) / DH];
    }
    if (k0 + lane >= n_keys) s = -INFINITY;
    const float mn = fmaxf(m, wave_max(s));
    const float alpha = m == mn ? 1.f : fast_exp2(m - mn);
    const float p = s == -INFINITY && mn == s ? 0.f : fast_exp2(s - mn);
    l = l * alpha + wave_sum(p);
    m = mn;
#pragma unroll
    for (int i = 0; i < DH / 64; ++i) acc[i] *= alpha;
#pragma unroll 1
    for (int u = 0; u < min(64, n_keys - k0); ++u) {
      const float pu = __shfl(p * vs, u, 64);
      const int64_t vu = __shfl(at, u, 64);
#pragma unroll
      for (int i = 0; i < DH / 64; ++i) acc[i] += pu * to_float(vc[vu + lane + 64 * i]);
    }
  }
  float *out = static_cast<float *>(a.out) + (int64_t)token * a.o_ts + (int64_t)qh * a.o_hs;
#pragma unroll
  for (int i = 0; i < DH / 64; ++i)
    out[lane + 64 * i] = n_keys > 0 ? acc[i] / l * a.v_scale : 0.f;
}

// At most 256 registers (at Dh 128 two workgroups fit a CU's LDS).
template <typename KV, int DH, bool ROWS>
__global__ __launch_bounds__(64 * kFWaves) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_f32_kernel(PrefillArgs a, int G) {
  constexpr int QC = DH / 16;  // 16-byte chunks of a row per lane
  constexpr int VC = DH / 64;  // 64-dim groups
  constexpr int LD = DH + 4;
  typedef RowPart<KV, DH> Part;
  __shared__ __attribute__((aligned(16))) float k_s[2][kFKeys][LD];
  __shared__ __attribute__((aligned(16))) float v_s[2][kFKeys][LD];
  __shared__ __attribute__((aligned(16))) float ks_s[2][ROWS ? kFKeys : 4];
  __shared__ __attribute__((aligned(16))) float vs_s[2][ROWS ? kFKeys : 4];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int r = lane & 15;
  const int g = lane >> 4;

  // Up to 64 sequences: the tiles with most keys first (workgroups of one tile, one per KV
  // head, follow each other). Larger batches: every sequence's last tile first, then the
  // one before; the pairs move on by one per tile, so that no XCD (workgroup i runs on XCD
  // i % 8) keeps the longest sequences.
  const int QT = kFRows / G;  // query tokens per workgroup (rows from QT * G on are unused)
  int b, tile, kvh;
  if (a.num_seqs <= kTileOrderSeqs) {
    QueryTile qt;
    if (!find_query_tile(a.cu_q, a.seq_lens, a.num_seqs, QT, (a.key_cap + QT - 1) / QT,
                         blockIdx.x / a.num_kv_heads, lane, &qt))
      return;
    b = __builtin_amdgcn_readfirstlane(qt.seq);
    tile = __builtin_amdgcn_readfirstlane(qt.tile);
    kvh = blockIdx.x % a.num_kv_heads;
  } else {
    const int level = blockIdx.x / a.num_pairs;
    const int pair = (blockIdx.x + level) % a.num_pairs;
    tile = a.tiles - 1 - level;
    kvh = pair % a.num_kv_heads;
    const int rank = pair / a.num_kv_heads;
    b = a.seq_order ? min(max(a.seq_order[rank], 0), a.num_seqs - 1) : rank;
  }
  const int q0 = a.cu_q[b];
  const int q_len = a.cu_q[b + 1] - q0;
  const int t0 = tile * QT;
  if (t0 >= q_len) return;
  const int base_pos = a.seq_lens[b] - q_len;  // position of query token 0
  const int t_end = min(q_len, t0 + QT);
  const int n_keys = max(0, min(base_pos + t_end, a.key_cap));
  const int n_steps = (n_keys + kFKeys - 1) / kFKeys;

  const float *q = static_cast<const float *>(a.q);
  const int64_t head_base = a.pool.layer_base + (int64_t)kvh * a.pool.head_stride;
  const KV *kc = static_cast<const KV *>(a.kc) + head_base;
  const KV *vc = static_cast<const KV *>(a.vc) + head_base;
  const int32_t *bt_row = a.bt + (int64_t)b * a.bt_stride;
  const int BS = a.pool.block_size;

  // Staging: thread tid loads part tid % 8 of row tid / 8 of a step. Its key of the step to
  // load next is row s_in of block s_blk of the sequence, whose id is read one step ahead.
  const int s_row = tid >> 3, s_c = tid & 7;
  int s_blk = s_row / BS, s_in = s_row % BS;
  auto block_at = [&](int step) -> int64_t {
    return step * kFKeys + s_row < n_keys ? block_of(bt_row, s_blk, a.pool.num_blocks) : 0;
  };
  int64_t blk_next = block_at(0);
  Part kp, vp;
  float ksv = 0.f, vsv = 0.f;
  auto load_rows = [&](int step) {
    const int key = step * kFKeys + s_row;
    if (key < n_keys) {
      const int64_t at = blk_next * a.pool.block_stride + s_in * DH;
      kp.load(kc + at, s_c);
      vp.load(vc + at, s_c);
      if constexpr (ROWS) {
        ksv = a.k_rs[(head_base + at) / DH];
        vsv = a.v_rs[(head_base + at) / DH];
      }
    } else {  // past the last key: scores are masked, and 0 * V must not be NaN
      kp.zero();
      vp.zero();
      ksv = vsv = 0.f;
    }
    for (s_in += kFKeys; s_in >= BS; s_in -= BS) ++s_blk;
    blk_next = block_at(step + 1);
  };
  auto store_rows = [&](auto slot_c) {
    constexpr int buf = decltype(slot_c)::value;
    kp.store(&k_s[buf][s_row][0], s_c);
    vp.store(&v_s[buf][s_row][0], s_c);
    if constexpr (ROWS) {
      if (s_c == 0) {
        ks_s[buf][s_row] = ksv;
        vs_s[buf][s_row] = vsv;
      }
    }
  };
  load_rows(0);  // (a step past the last loads nothing)

  // Q^T operands of row wave * 16 + r. qpos: the last key it sees (-1: none, or padding).
  const int row = wave * 16 + r;
  const int token = t0 + row / G, head = kvh * G + row % G;
  const bool in = row < QT * G && token < t_end;
  const int qpos = in ? max(-1, min(base_pos + token, a.key_cap - 1)) : -1;
  const int min_pos = __reduce_min_sync(~0ull, in ? qpos : 0x7fffffff);
  const float *qp = q + (int64_t)(q0 + min(token, q_len - 1)) * a.q_ts + (int64_t)head * a.q_hs;
  f32x4 qf[QC];
#pragma unroll
  for (int c = 0; c < QC; ++c)
    qf[c] = in ? *reinterpret_cast<const f32x4 *>(qp + 16 * c + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};

  f32x4 acc[4 * VC];
  // Online softmax of row r, in log2 units: m the reference maximum (it moves when a score
  // passes it by more than 8), l this lane's share of the sum.
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int d = 0; d < 4 * VC; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float scale_log2 = a.scale_log2;  // > 0 (the host routes other scales elsewhere)

  store_rows(Slot<0>{});
  __syncthreads();

  auto step = [&](auto slot_c, int s) {
    constexpr int buf = decltype(slot_c)::value;
    load_rows(s + 1);
    const int k0 = s * kFKeys;

    f32x4 st[2] = {};
#pragma unroll
    for (int c = 0; c < QC; ++c) {
      f32x4 kf[2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        kf[kt] = *reinterpret_cast<const f32x4 *>(&k_s[buf][kt * 16 + r][16 * c + 4 * g]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) st[kt] = mfma_f32(kf[kt][e], qf[c][e], st[kt]);
    }
    f32x4 vs4[2];
    if constexpr (ROWS) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const f32x4 ks4 = *reinterpret_cast<const f32x4 *>(&ks_s[buf][kt * 16 + 4 * g]);
        vs4[kt] = *reinterpret_cast<const f32x4 *>(&vs_s[buf][kt * 16 + 4 * g]);
        st[kt] *= ks4;
      }
    }
    // Steps past the wave's first query position: key k0 + kt*16 + 4g + i is seen iff it
    // is <= qpos (which also keeps it below n_keys).
    const bool need_mask = k0 + kFKeys - 1 > min_pos;
    if (need_mask) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (k0 + kt * 16 + 4 * g + i > qpos) st[kt][i] = -INFINITY;
    }
    const float a0 = nan_max(nan_max(st[0][0], st[0][1]), nan_max(st[0][2], st[0][3]));
    const float a1 = nan_max(nan_max(st[1][0], st[1][1]), nan_max(st[1][2], st[1][3]));
    const float lm = nan_max(a0, a1) * scale_log2;
    if (__builtin_amdgcn_ballot_w64(lm > m + 8.f)) {
      const float mx = xgroup_max(lm);
      const bool bump = mx > m + 8.f;
      const float alpha = bump ? fast_exp2(m - mx) : 1.f;
      m = bump ? mx : m;
      l *= alpha;
#pragma unroll
      for (int d = 0; d < 4 * VC; ++d) acc[d] *= alpha;
    }
    const float nr = m == -INFINITY ? 0.f : -m;
    float sum[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        st[kt][i] = fast_exp2(__builtin_fmaf(st[kt][i], scale_log2, nr));
      sum[kt] = (st[kt][0] + st[kt][1]) + (st[kt][2] + st[kt][3]);
    }
    l += sum[0] + sum[1];
    if constexpr (ROWS) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) st[kt] *= vs4[kt];
    }

    auto v_operand = [&](int kt, int i, int h) {
      return *reinterpret_cast<const float4 *>(&v_s[buf][kt * 16 + 4 * g + i][64 * h + 4 * r]);
    };
    // The step's sums start from zero and are added to the row's: shorter chains of
    // roundings than one over all keys (error of the prompts above against 64 bits
    // 2.1e-7, 2.5e-7 with one; the VALU kernel's is 2.3e-7).
#pragma unroll
    for (int h = 0; h < VC; ++h) {
      f32x4 o[4] = {};
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float4 vf = v_operand(kt, i, h);
          o[0] = mfma_f32(vf.x, st[kt][i], o[0]);
          o[1] = mfma_f32(vf.y, st[kt][i], o[1]);
          o[2] = mfma_f32(vf.z, st[kt][i], o[2]);
          o[3] = mfma_f32(vf.w, st[kt][i], o[3]);
        }
#pragma unroll
      for (int d = 0; d < 4; ++d) acc[4 * h + d] += o[d];
      register_fence<DH>();
    }
    store_rows(Slot<buf ^ 1>{});
    __syncthreads();
  };
  for (int s = 0; s < n_steps; s += 2) {
    step(Slot<0>{}, s);
    if (s + 1 < n_steps) step(Slot<1>{}, s + 1);
  }

  // A V value (or row scale) that is not finite, under a key that some rows of a tile do
  // not see, has reached those rows too (0 * inf is NaN): a wave whose sums are not all
  // finite takes its rows one by one.
  float bad = 0.f;
#pragma unroll
  for (int d = 0; d < 4 * VC; ++d)
#pragma unroll
    for (int i = 0; i < 4; ++i) bad += 0.f * acc[d][i];
  if (__builtin_amdgcn_ballot_w64(bad != bad)) {
#pragma unroll 1
    for (int k = 0; k < 16; ++k) {
      const int x = wave * 16 + k, t = t0 + x / G;
      if (x < QT * G && t < t_end)
        one_row<KV, DH>(a, kvh * G + x % G, kc, vc, head_base, bt_row, q0 + t,
                        max(0, min(base_pos + t + 1, a.key_cap)), lane);
    }
    return;
  }

  // Lane (g, r) holds dims 64 h + 16 g + 4 i + d of row r in acc[4 h + d][i].
  float *out = static_cast<float *>(a.out);
  l = xgroup_sum(l);
  if (!in) return;
  const bool any = qpos >= 0;  // a row without keys is zero
  float *op = out + (int64_t)(q0 + token) * a.o_ts + (int64_t)head * a.o_hs + 16 * g;
#pragma unroll
  for (int c = 0; c < VC; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float o[4];
#pragma unroll
      for (int d = 0; d < 4; ++d) o[d] = any ? acc[4 * c + d][i] / l * a.v_scale : 0.f;
      *reinterpret_cast<float4 *>(op + 64 * c + 4 * i) = make_float4(o[0], o[1], o[2], o[3]);
    }
}

template <typename KV, bool ROWS>
int32_t launch_f32(const PrefillArgs &a, int32_t G, int32_t head_dim, dim3 grid, hipStream_t s) {
  if (head_dim == 64)
    prefill_f32_kernel<KV, 64, ROWS><<<grid, 64 * kFWaves, 0, s>>>(a, G);
  else
    prefill_f32_kernel<KV, 128, ROWS><<<grid, 64 * kFWaves, 0, s>>>(a, G);
  return check_launch();
}

int64_t prefill_f32_blocks(int64_t num_seqs, int64_t num_tokens, int64_t num_kv_heads, int32_t group,
                           int64_t max_query_len) {
  const int64_t qt = kFRows / group;
  // Tiles of n sequences with N tokens in all: at most N / QT + n. (A chunk longer than the
  // batch's tokens does not exist: max_query_len may be a loose bound.)
  return num_seqs <= kTileOrderSeqs
             ? (num_tokens / qt + num_seqs) * num_kv_heads
             : num_seqs * num_kv_heads * ceil_div(std::min(max_query_len, num_tokens), qt);
}

}  // namespace

bool prefill_f32_supported(int32_t head_dim, int32_t group, int64_t num_seqs, int64_t num_tokens,
                           int64_t num_kv_heads, int64_t max_query_len) {
  return (head_dim == 64 || head_dim == 128) && group >= 1 && group <= 16 &&
         num_seqs * num_kv_heads <= INT32_MAX &&
         // A launch has fewer than 2^32 threads.
         prefill_f32_blocks(num_seqs, num_tokens, num_kv_heads, group, max_query_len) <
             (int64_t{1} << 32) / (64 * kFWaves);
}

int32_t launch_prefill_f32(const PrefillArgs &a, int32_t num_seqs, int64_t num_tokens,
                           int32_t num_kv_heads, int32_t group, int32_t head_dim,
                           int32_t max_query_len, bool fp8_pools, hipStream_t stream) {
  PrefillArgs args = a;
  args.num_kv_heads = num_kv_heads;
  args.num_seqs = num_seqs;
  args.num_pairs = num_seqs * num_kv_heads;
  args.tiles = static_cast<int32_t>(
      ceil_div(std::min<int64_t>(max_query_len, num_tokens), kFRows / group));
  if (args.tiles == 0 || args.num_pairs == 0) return TKS_OK;
  const int64_t blocks =
      prefill_f32_blocks(num_seqs, num_tokens, num_kv_heads, group, max_query_len);
  const dim3 grid(static_cast<unsigned>(blocks));
  if (!fp8_pools) return launch_f32<float, false>(args, group, head_dim, grid, stream);
  return a.k_rs != nullptr ? launch_f32<fp8e4m3_t, true>(args, group, head_dim, grid, stream)
                           : launch_f32<fp8e4m3_t, false>(args, group, head_dim, grid, stream);
}

}  // namespace tks
