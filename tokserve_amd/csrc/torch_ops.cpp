// Device kernels of the operators an iteration calls, registered with the dispatcher
// from here: the addresses, strides and stream go to the C entry points without passing
// through Python (torch_ops.py declares the schemas and fake kernels, and keeps the other
// operators' device kernels). Small calls last as long as the host takes for them: the
// fused decode of 8 sequences 20.6 us through the ctypes binding and 12.5 us from here, the
// greedy choice of 16 rows 10.6 and 6.8 us, a 1.1B model's iteration (about 200 calls)
// 5,060 and 4,000 us.
//
// The entry points are looked up in libtokserve_hip.so on the first call, so loading this
// library does not touch HIP. It is loaded and registered by torch_ops.py, which first
// compares the versions it was built against (of torch, and of the C ABI that it calls
// through) with those it is loaded into. Errors are raised by tokserve_amd.kernels._lib, which maps a
// status to its exception.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/library.h>
#include <torch/headeronly/version.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <dlfcn.h>

#include <atomic>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>

#include "tokserve_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

#define TKS_ENTRY_POINTS(X)              \
  X(tks_paged_attention_decode_workspace_bytes) \
  X(tks_paged_attention_decode)          \
  X(tks_paged_attention_decode_fp8)      \
  X(tks_paged_attention_decode_fp8_rows) \
  X(tks_paged_attention_prefill)         \
  X(tks_paged_attention_prefill_fp8_workspace_bytes) \
  X(tks_paged_attention_prefill_fp8)     \
  X(tks_paged_attention_prefill_fp8_rows) \
  X(tks_rope_append_paged_decode)        \
  X(tks_rope_append_paged_decode_fp8)    \
  X(tks_rope_append_paged_decode_fp8_rows) \
  X(tks_rope_kv_append)                  \
  X(tks_rope_kv_append_fp8)              \
  X(tks_rope_kv_append_fp8_rows)         \
  X(tks_rms_norm)                        \
  X(tks_argmax)                          \
  X(tks_silu_mul)

struct Library {
#define TKS_FIELD(name) decltype(&::name) name = nullptr;
  TKS_ENTRY_POINTS(TKS_FIELD)
#undef TKS_FIELD
};

// f() with the GIL held, its exception passed on as a kernel in Python would raise it.
template <typename F>
auto with_python(F f) {
  pybind11::gil_scoped_acquire gil;
  try {
    return f();
  } catch (pybind11::error_already_set &raised) {
    raised.restore();
    python_error error;
    error.persist();
    throw error;
  }
}

// The library _lib.load() loads (and checks).
Library look_up() {
  const std::string path = with_python([] {
    pybind11::module_ lib = pybind11::module_::import("tokserve_amd.kernels._lib");
    lib.attr("load")();
    return std::string(pybind11::str(lib.attr("library_path")()));
  });
  void *handle = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  if (handle == nullptr) throw std::runtime_error(dlerror());
  Library l;
#define TKS_LOOK_UP(name)                                            \
  l.name = reinterpret_cast<decltype(l.name)>(dlsym(handle, #name)); \
  if (l.name == nullptr) throw std::runtime_error(std::string("missing ") + #name);
  TKS_ENTRY_POINTS(TKS_LOOK_UP)
#undef TKS_LOOK_UP
  return l;
}

const Library &library() {
  static std::atomic<const Library *> ready{nullptr};
  if (const Library *l = ready.load(std::memory_order_acquire)) return *l;
  // Without the GIL, which look_up() takes under the lock of the static below.
  std::optional<pybind11::gil_scoped_release> released;
  if (PyGILState_Check()) released.emplace();
  static const Library loaded = look_up();
  ready.store(&loaded, std::memory_order_release);
  return loaded;
}

void check(int32_t status, const char *operation) {
  if (status == TKS_OK) return;
  with_python([&] {
    return pybind11::module_::import("tokserve_amd.kernels._lib").attr("check")(status, operation)
        .is_none();  // (raises)
  });
}

int32_t code(const Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return TKS_FLOAT32;
    case at::kHalf: return TKS_FLOAT16;
    case at::kBFloat16: return TKS_BFLOAT16;
    default: break;
  }
  return with_python([&] {
    return pybind11::module_::import("tokserve_amd.kernels._lib")
        .attr("dtype_code")(pybind11::handle(
            reinterpret_cast<PyObject *>(torch::getTHPDtype(t.scalar_type()))))
        .cast<int32_t>();  // (raises)
  });
}

tks_stream_t stream_of(const Tensor &t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

const void *ptr(const OptTensor &t) { return t ? t->const_data_ptr() : nullptr; }
void *mut(const OptTensor &t) { return t ? t->mutable_data_ptr() : nullptr; }
template <typename T>
T *as(const Tensor &t) { return static_cast<T *>(t.mutable_data_ptr()); }
template <typename T>
T *as(const OptTensor &t) { return static_cast<T *>(mut(t)); }
int32_t i32(int64_t x) { return static_cast<int32_t>(x); }
bool fp8(const Tensor &pool) { return pool.scalar_type() == at::kFloat8_e4m3fn; }

// Scratch memory of one call, undefined for 0 bytes: from the caching allocator on the
// launch's stream, so no other call, stream or thread shares it.
Tensor scratch(int64_t bytes, const Tensor &query, const char *use) {
  TORCH_CHECK_VALUE(bytes >= 0, "invalid ", use, " workspace query");
  return bytes == 0 ? Tensor() : at::empty({bytes}, query.options().dtype(at::kByte));
}

// Split partials of a decode: the caller's workspace, or scratch.
Tensor decode_workspace(const OptTensor &given, const Tensor &query, const Tensor &pool,
                        int64_t max_seq_len, int64_t pages_per_split) {
  if (given) return *given;
  return scratch(library().tks_paged_attention_decode_workspace_bytes(
                     i32(query.size(0)), i32(query.size(1)), i32(pool.size(2)), i32(pool.size(4)),
                     i32(pool.size(3)), i32(max_seq_len), i32(pages_per_split)),
                 query, "decode");
}

void paged_attention_decode(const Tensor &query, const Tensor &key_cache,
                            const Tensor &value_cache, const Tensor &block_tables,
                            const Tensor &seq_lens, const OptTensor &seq_order,
                            int64_t layer_index, int64_t max_seq_len, double scale,
                            int64_t pages_per_split, double k_scale, double v_scale,
                            const Tensor &out, const OptTensor &workspace,
                            const OptTensor &k_scales, const OptTensor &v_scales) {
  const Library &l = library();
  const Tensor ws = decode_workspace(workspace, query, key_cache, max_seq_len, pages_per_split);
  void *ws_ptr = ws.defined() ? ws.mutable_data_ptr() : nullptr;
  const int64_t ws_bytes = ws.defined() ? ws.numel() : 0;
  const Tensor &kc = key_cache;
  auto call = [&](auto entry, auto scales, auto... factors) {
    return std::apply(
        [&](auto... rows) {
          return entry(query.const_data_ptr(), query.stride(0), query.stride(1),
                       kc.const_data_ptr(), value_cache.const_data_ptr(), rows...,
                       i32(kc.size(0)), kc.size(1), i32(kc.size(2)), i32(kc.size(3)),
                       i32(kc.size(4)), i32(layer_index), as<int32_t>(block_tables),
                       i32(block_tables.size(1)), as<int32_t>(seq_lens), as<int32_t>(seq_order),
                       i32(query.size(0)), i32(query.size(1)), i32(max_seq_len),
                       static_cast<float>(scale), i32(pages_per_split), out.mutable_data_ptr(),
                       out.stride(0), out.stride(1), ws_ptr, ws_bytes, factors..., code(query),
                       stream_of(query));
        },
        scales);
  };
  const auto none = std::tuple<>();
  check(k_scales ? call(l.tks_paged_attention_decode_fp8_rows,
                        std::make_tuple(as<const float>(k_scales), as<const float>(v_scales)))
        : fp8(kc) ? call(l.tks_paged_attention_decode_fp8, none, static_cast<float>(k_scale),
                         static_cast<float>(v_scale))
                  : call(l.tks_paged_attention_decode, none),
        "paged_attention_decode");
}

// The decoded pages of fp8 pools.
Tensor fp8_pages(const Tensor &query, const Tensor &pool, int64_t num_seqs, int64_t table_width,
                 int64_t max_seq_len) {
  return scratch(library().tks_paged_attention_prefill_fp8_workspace_bytes(
                     i32(num_seqs), i32(query.size(1)), i32(pool.size(2)), i32(pool.size(4)),
                     i32(pool.size(3)), i32(table_width), i32(max_seq_len), code(query)),
                 query, "fp8 prefill");
}

void paged_attention_prefill(const Tensor &query, const Tensor &key_cache,
                             const Tensor &value_cache, const Tensor &block_tables,
                             const Tensor &seq_lens, const Tensor &cu_seqlens_q,
                             const OptTensor &seq_order, int64_t layer_index,
                             int64_t max_query_len, int64_t max_seq_len, double scale,
                             double k_scale, double v_scale, const Tensor &out,
                             const OptTensor &k_scales, const OptTensor &v_scales) {
  const Library &l = library();
  const Tensor &kc = key_cache;
  auto call = [&](auto entry, auto scales, auto... tail) {
    return std::apply(
        [&](auto... rows) {
          return entry(query.const_data_ptr(), query.stride(0), query.stride(1),
                       kc.const_data_ptr(), value_cache.const_data_ptr(), rows...,
                       i32(kc.size(0)), kc.size(1), i32(kc.size(2)), i32(kc.size(3)),
                       i32(kc.size(4)), i32(layer_index), as<int32_t>(block_tables),
                       i32(block_tables.size(1)), as<int32_t>(seq_lens),
                       as<int32_t>(cu_seqlens_q), as<int32_t>(seq_order), i32(seq_lens.size(0)),
                       query.size(0), i32(query.size(1)), i32(max_query_len), i32(max_seq_len),
                       static_cast<float>(scale), out.mutable_data_ptr(), out.stride(0),
                       out.stride(1), tail..., code(query), stream_of(query));
        },
        scales);
  };
  const auto none = std::tuple<>();
  int32_t status;
  if (fp8(kc)) {
    const Tensor ws =
        fp8_pages(query, kc, seq_lens.size(0), block_tables.size(1), max_seq_len);
    void *ws_ptr = ws.defined() ? ws.mutable_data_ptr() : nullptr;
    const int64_t ws_bytes = ws.defined() ? ws.numel() : 0;
    status = k_scales ? call(l.tks_paged_attention_prefill_fp8_rows,
                             std::make_tuple(as<const float>(k_scales), as<const float>(v_scales)),
                             ws_ptr, ws_bytes)
                      : call(l.tks_paged_attention_prefill_fp8, none, ws_ptr, ws_bytes,
                             static_cast<float>(k_scale), static_cast<float>(v_scale));
  } else {
    status = call(l.tks_paged_attention_prefill, none);
  }
  check(status, "paged_attention_prefill");
}

void rope_append_paged_decode(
    const Tensor &query, const Tensor &key, const Tensor &value, const Tensor &positions,
    const Tensor &cos, const Tensor &sin, const Tensor &slot_mapping, const Tensor &key_cache,
    const Tensor &value_cache, const Tensor &block_tables, const Tensor &seq_lens,
    const OptTensor &seq_order, int64_t layer_index, int64_t max_seq_len, double scale,
    int64_t pages_per_split, const Tensor &out, const OptTensor &workspace, double k_scale,
    double v_scale, const OptTensor &k_scales, const OptTensor &v_scales) {
  const Library &l = library();
  const Tensor ws = decode_workspace(workspace, query, key_cache, max_seq_len, pages_per_split);
  void *ws_ptr = ws.defined() ? ws.mutable_data_ptr() : nullptr;
  const int64_t ws_bytes = ws.defined() ? ws.numel() : 0;
  const Tensor &kc = key_cache;
  auto call = [&](auto entry, auto scales, auto... factors) {
    return std::apply(
        [&](auto... rows) {
          return entry(query.const_data_ptr(), query.stride(0), query.stride(1),
                       key.const_data_ptr(), key.stride(0), key.stride(1),
                       value.const_data_ptr(), value.stride(0), value.stride(1),
                       as<int64_t>(positions), cos.const_data_ptr(), sin.const_data_ptr(),
                       cos.size(0), as<int64_t>(slot_mapping), kc.mutable_data_ptr(),
                       value_cache.mutable_data_ptr(), rows..., i32(kc.size(0)), kc.size(1),
                       i32(kc.size(2)), i32(kc.size(3)), i32(kc.size(4)), i32(layer_index),
                       as<int32_t>(block_tables), i32(block_tables.size(1)),
                       as<int32_t>(seq_lens), as<int32_t>(seq_order), i32(query.size(0)),
                       i32(query.size(1)), i32(max_seq_len), static_cast<float>(scale),
                       i32(pages_per_split), out.mutable_data_ptr(), out.stride(0),
                       out.stride(1), ws_ptr, ws_bytes, factors..., code(query),
                       stream_of(query));
        },
        scales);
  };
  const auto none = std::tuple<>();
  check(k_scales ? call(l.tks_rope_append_paged_decode_fp8_rows,
                        std::make_tuple(as<float>(k_scales), as<float>(v_scales)))
        : fp8(kc) ? call(l.tks_rope_append_paged_decode_fp8, none, static_cast<float>(k_scale),
                         static_cast<float>(v_scale))
                  : call(l.tks_rope_append_paged_decode, none),
        "rope_append_paged_decode");
}

void rope_kv_append(const Tensor &query, const Tensor &key, const Tensor &value,
                    const Tensor &positions, const Tensor &cos, const Tensor &sin,
                    const Tensor &key_cache, const Tensor &value_cache,
                    const Tensor &slot_mapping, int64_t layer_index, const Tensor &query_out,
                    const OptTensor &key_out, double k_scale, double v_scale,
                    const OptTensor &k_scales, const OptTensor &v_scales) {
  const Library &l = library();
  const Tensor &kc = key_cache;
  auto call = [&](auto entry, auto scales, auto... factors) {
    return std::apply(
        [&](auto... rows) {
          return entry(query.const_data_ptr(), query_out.mutable_data_ptr(), query.stride(0),
                       query.stride(1), query_out.stride(0), query_out.stride(1),
                       i32(query.size(1)), key.const_data_ptr(), mut(key_out), key.stride(0),
                       key.stride(1), key_out ? key_out->stride(0) : 0,
                       key_out ? key_out->stride(1) : 0, value.const_data_ptr(),
                       value.stride(0), value.stride(1), i32(kc.size(2)), query.size(0),
                       i32(kc.size(4)), as<int64_t>(positions), cos.const_data_ptr(),
                       sin.const_data_ptr(), cos.size(0), kc.mutable_data_ptr(),
                       value_cache.mutable_data_ptr(), rows..., i32(kc.size(0)), kc.size(1),
                       i32(kc.size(3)), i32(layer_index), as<int64_t>(slot_mapping), factors...,
                       code(query), stream_of(query));
        },
        scales);
  };
  const auto none = std::tuple<>();
  check(k_scales ? call(l.tks_rope_kv_append_fp8_rows,
                        std::make_tuple(as<float>(k_scales), as<float>(v_scales)))
        : fp8(kc) ? call(l.tks_rope_kv_append_fp8, none, static_cast<float>(k_scale),
                         static_cast<float>(v_scale))
                  : call(l.tks_rope_kv_append, none),
        "rope_kv_append");
}

void rope_kv_append_(const Tensor &query, const Tensor &key, const Tensor &value,
                     const Tensor &positions, const Tensor &cos, const Tensor &sin,
                     const Tensor &key_cache, const Tensor &value_cache,
                     const Tensor &slot_mapping, int64_t layer_index, const OptTensor &key_out,
                     double k_scale, double v_scale, const OptTensor &k_scales,
                     const OptTensor &v_scales) {
  rope_kv_append(query, key, value, positions, cos, sin, key_cache, value_cache, slot_mapping,
                 layer_index, query, key_out, k_scale, v_scale, k_scales, v_scales);
}

void rms_norm(const Tensor &input, const Tensor &weight, double epsilon,
              const OptTensor &residual, const Tensor &out, const OptTensor &residual_out) {
  check(library().tks_rms_norm(
            input.const_data_ptr(), input.stride(0), ptr(residual),
            residual ? residual->stride(0) : 0, mut(residual_out),
            residual_out ? residual_out->stride(0) : 0, weight.const_data_ptr(),
            out.mutable_data_ptr(), out.stride(0), input.size(0), i32(input.size(1)),
            static_cast<float>(epsilon), code(input), code(weight), code(out), stream_of(input)),
        "rms_norm");
}

void greedy_argmax(const Tensor &logits, const Tensor &out) {
  check(library().tks_argmax(logits.const_data_ptr(), logits.stride(0), logits.size(0),
                             logits.size(1), as<int64_t>(out), code(logits), stream_of(logits)),
        "greedy_argmax");
}

void silu_mul(const Tensor &gate_up, const Tensor &out) {
  check(library().tks_silu_mul(gate_up.const_data_ptr(), gate_up.stride(0), gate_up.size(0),
                               gate_up.size(1) / 2, out.mutable_data_ptr(), out.stride(0),
                               code(gate_up), stream_of(gate_up)),
        "silu_mul");
}

}  // namespace

extern "C" const char *tks_torch_built_for(void) { return TORCH_VERSION; }

extern "C" int32_t tks_torch_abi_version(void) { return TKS_ABI_VERSION; }

// Registers the device kernels, once; null, or why not.
extern "C" const char *tks_torch_register(void) {
  static std::string error;
  try {
    static const torch::Library kernels = [] {
      torch::Library m(torch::Library::IMPL, "tokserve_amd", c10::DispatchKey::CUDA, __FILE__,
                       __LINE__);
      m.impl("paged_attention_decode", paged_attention_decode);
      m.impl("paged_attention_prefill", paged_attention_prefill);
      m.impl("rope_append_paged_decode", rope_append_paged_decode);
      m.impl("rope_kv_append", rope_kv_append);
      m.impl("rope_kv_append_", rope_kv_append_);
      m.impl("rms_norm", rms_norm);
      m.impl("greedy_argmax", greedy_argmax);
      m.impl("silu_mul", silu_mul);
      return m;
    }();
  } catch (const std::exception &raised) {
    error = raised.what();
    return error.c_str();
  }
  return nullptr;
}
