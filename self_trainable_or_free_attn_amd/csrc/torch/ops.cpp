// Generated by self_trainable_or_free_attn_amd/torch_ops.py from include/echosparse_hip.h and
// include/vsa_hip.h: one torch operator per stream-taking C entry point. Do not edit by hand.
#include "../../../include/vsa_hip.h"

#include <ATen/core/Tensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <cstdint>
#include <initializer_list>

namespace {

// the device, guard and current stream of a call; refuses host tensors and tensors on two devices
struct Call {
  const char* name;
  c10::optional<c10::Device> dev;
  Call(const char* n, std::initializer_list<const c10::optional<at::Tensor>*> ts) : name(n) {
    for (const auto* t : ts) {
      if (!t->has_value()) continue;
      const at::Tensor& x = **t;
      TORCH_CHECK(x.is_cuda(), name, ": every tensor argument must live on the GPU (got a ", x.device(),
                  " tensor)");
      if (!dev) dev = x.device();
      TORCH_CHECK(x.device() == *dev, name, ": tensors on two devices (", *dev, " and ", x.device(), ")");
    }
  }
};

enum EsDtype { ES_F32, ES_I32, ES_U8, ES_HALF, ES_OUT, ES_ANY };

// the pointer of an optional tensor argument after checking its layout and its dtype against the C type
inline void* es_op_data(const char* name, const char* arg, const c10::optional<at::Tensor>& t, EsDtype kind) {
  if (!t.has_value()) return nullptr;
  const at::Tensor& x = *t;
  TORCH_CHECK(x.is_contiguous(), name, ": argument ", arg, " must be contiguous");
  const at::ScalarType s = x.scalar_type();
  bool ok = true;
  const char* want = "";
  switch (kind) {
    case ES_F32: ok = s == at::kFloat; want = "float32"; break;
    case ES_I32: ok = s == at::kInt || s == at::kUInt32; want = "int32"; break;
    case ES_U8: ok = s == at::kByte || s == at::kBool; want = "uint8"; break;
    case ES_HALF: ok = s == at::kBFloat16 || s == at::kHalf; want = "bfloat16 or float16"; break;
    case ES_OUT:
      ok = s == at::kBFloat16 || s == at::kHalf || s == at::kFloat;
      want = "bfloat16, float16 or float32";
      break;
    case ES_ANY: break;
  }
  TORCH_CHECK(ok, name, ": argument ", arg, " must be ", want, " (got ", s, ")");
  return x.data_ptr();
}

enum EsInt { ES_INT, ES_UINT, ES_SIZE, ES_LL };

// an integer argument, refused if it does not fit the C parameter type
inline int64_t es_op_int(const char* name, const char* arg, int64_t v, EsInt kind) {
  const bool ok = kind == ES_INT    ? v >= INT32_MIN && v <= INT32_MAX
                : kind == ES_UINT   ? v >= 0 && v <= int64_t(UINT32_MAX)
                : kind == ES_SIZE   ? v >= 0
                                    : true;
  TORCH_CHECK(ok, name, ": argument ", arg, " = ", v, " is out of range for its C type");
  return v;
}

inline void es_op_check(const char* name, int status) {
  TORCH_CHECK(status == 0, name, " failed (status ", status, "): ", es_last_error_string());
}

}  // namespace

static void op_es_block_attention(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& blocks, int64_t nk, const c10::optional<at::Tensor>& offset, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& flags, const c10::optional<at::Tensor>& mass, double threshold, int64_t L, int64_t H, int64_t D) {
  const Call es_op_call("es_block_attention", {&q, &k, &v, &out, &counts, &blocks, &offset, &lse, &flags, &mass});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_block_attention", es_block_attention(static_cast<const void*>(es_op_data("es_block_attention", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("es_block_attention", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("es_block_attention", "v", v, ES_HALF)), static_cast<void*>(es_op_data("es_block_attention", "out", out, ES_OUT)), static_cast<const int*>(es_op_data("es_block_attention", "counts", counts, ES_I32)), static_cast<const int*>(es_op_data("es_block_attention", "blocks", blocks, ES_I32)), static_cast<int>(es_op_int("es_block_attention", "nk", nk, ES_INT)), static_cast<const float*>(es_op_data("es_block_attention", "offset", offset, ES_F32)), static_cast<float*>(es_op_data("es_block_attention", "lse", lse, ES_F32)), static_cast<int*>(es_op_data("es_block_attention", "flags", flags, ES_I32)), static_cast<float*>(es_op_data("es_block_attention", "mass", mass, ES_F32)), static_cast<float>(threshold), static_cast<int>(es_op_int("es_block_attention", "L", L, ES_INT)), static_cast<int>(es_op_int("es_block_attention", "H", H, ES_INT)), static_cast<int>(es_op_int("es_block_attention", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_block_attention(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& blocks, int64_t nk, const c10::optional<at::Tensor>& offset, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& flags, const c10::optional<at::Tensor>& mass, double threshold, int64_t L, int64_t H, int64_t D) {}

static void op_es_sparse_attention(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& v_mean, const c10::optional<at::Tensor>& means, const c10::optional<at::Tensor>& mean_counts, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& blocks, int64_t nk, const c10::optional<at::Tensor>& offset, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& flags, const c10::optional<at::Tensor>& refine, const c10::optional<at::Tensor>& refine_counts, int64_t rw, const c10::optional<at::Tensor>& k_rep, const c10::optional<at::Tensor>& v_rep, const c10::optional<at::Tensor>& log_counts, const c10::optional<at::Tensor>& mass, double threshold, int64_t tiles, int64_t L, int64_t H, int64_t D) {
  const Call es_op_call("es_sparse_attention", {&q, &k, &v, &k_mean, &v_mean, &means, &mean_counts, &out, &counts, &blocks, &offset, &lse, &flags, &refine, &refine_counts, &k_rep, &v_rep, &log_counts, &mass});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_sparse_attention", es_sparse_attention(static_cast<const void*>(es_op_data("es_sparse_attention", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("es_sparse_attention", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("es_sparse_attention", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("es_sparse_attention", "k_mean", k_mean, ES_HALF)), static_cast<const void*>(es_op_data("es_sparse_attention", "v_mean", v_mean, ES_HALF)), static_cast<const int*>(es_op_data("es_sparse_attention", "means", means, ES_I32)), static_cast<const int*>(es_op_data("es_sparse_attention", "mean_counts", mean_counts, ES_I32)), static_cast<void*>(es_op_data("es_sparse_attention", "out", out, ES_OUT)), static_cast<const int*>(es_op_data("es_sparse_attention", "counts", counts, ES_I32)), static_cast<const int*>(es_op_data("es_sparse_attention", "blocks", blocks, ES_I32)), static_cast<int>(es_op_int("es_sparse_attention", "nk", nk, ES_INT)), static_cast<const float*>(es_op_data("es_sparse_attention", "offset", offset, ES_F32)), static_cast<float*>(es_op_data("es_sparse_attention", "lse", lse, ES_F32)), static_cast<int*>(es_op_data("es_sparse_attention", "flags", flags, ES_I32)), static_cast<const int*>(es_op_data("es_sparse_attention", "refine", refine, ES_I32)), static_cast<const int*>(es_op_data("es_sparse_attention", "refine_counts", refine_counts, ES_I32)), static_cast<int>(es_op_int("es_sparse_attention", "rw", rw, ES_INT)), static_cast<const void*>(es_op_data("es_sparse_attention", "k_rep", k_rep, ES_HALF)), static_cast<const void*>(es_op_data("es_sparse_attention", "v_rep", v_rep, ES_HALF)), static_cast<const float*>(es_op_data("es_sparse_attention", "log_counts", log_counts, ES_F32)), static_cast<float*>(es_op_data("es_sparse_attention", "mass", mass, ES_F32)), static_cast<float>(threshold), static_cast<int>(es_op_int("es_sparse_attention", "tiles", tiles, ES_INT)), static_cast<int>(es_op_int("es_sparse_attention", "L", L, ES_INT)), static_cast<int>(es_op_int("es_sparse_attention", "H", H, ES_INT)), static_cast<int>(es_op_int("es_sparse_attention", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_sparse_attention(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& v_mean, const c10::optional<at::Tensor>& means, const c10::optional<at::Tensor>& mean_counts, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& blocks, int64_t nk, const c10::optional<at::Tensor>& offset, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& flags, const c10::optional<at::Tensor>& refine, const c10::optional<at::Tensor>& refine_counts, int64_t rw, const c10::optional<at::Tensor>& k_rep, const c10::optional<at::Tensor>& v_rep, const c10::optional<at::Tensor>& log_counts, const c10::optional<at::Tensor>& mass, double threshold, int64_t tiles, int64_t L, int64_t H, int64_t D) {}

static void op_es_exact_fallback(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& blocks, int64_t nk, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& flags, int64_t L, int64_t H, int64_t D) {
  const Call es_op_call("es_exact_fallback", {&q, &k, &v, &out, &counts, &blocks, &lse, &flags});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_exact_fallback", es_exact_fallback(static_cast<const void*>(es_op_data("es_exact_fallback", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("es_exact_fallback", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("es_exact_fallback", "v", v, ES_HALF)), static_cast<void*>(es_op_data("es_exact_fallback", "out", out, ES_OUT)), static_cast<const int*>(es_op_data("es_exact_fallback", "counts", counts, ES_I32)), static_cast<const int*>(es_op_data("es_exact_fallback", "blocks", blocks, ES_I32)), static_cast<int>(es_op_int("es_exact_fallback", "nk", nk, ES_INT)), static_cast<float*>(es_op_data("es_exact_fallback", "lse", lse, ES_F32)), static_cast<const int*>(es_op_data("es_exact_fallback", "flags", flags, ES_I32)), static_cast<int>(es_op_int("es_exact_fallback", "L", L, ES_INT)), static_cast<int>(es_op_int("es_exact_fallback", "H", H, ES_INT)), static_cast<int>(es_op_int("es_exact_fallback", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_exact_fallback(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& blocks, int64_t nk, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& flags, int64_t L, int64_t H, int64_t D) {}

static void op_es_compensate_fallback(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& v_mean, const c10::optional<at::Tensor>& keep, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& flags, int64_t L, int64_t H, int64_t D) {
  const Call es_op_call("es_compensate_fallback", {&q, &k_mean, &v_mean, &keep, &lse, &out, &flags});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_compensate_fallback", es_compensate_fallback(static_cast<const void*>(es_op_data("es_compensate_fallback", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("es_compensate_fallback", "k_mean", k_mean, ES_HALF)), static_cast<const void*>(es_op_data("es_compensate_fallback", "v_mean", v_mean, ES_HALF)), static_cast<const uint8_t*>(es_op_data("es_compensate_fallback", "keep", keep, ES_U8)), static_cast<float*>(es_op_data("es_compensate_fallback", "lse", lse, ES_F32)), static_cast<void*>(es_op_data("es_compensate_fallback", "out", out, ES_OUT)), static_cast<const int*>(es_op_data("es_compensate_fallback", "flags", flags, ES_I32)), static_cast<int>(es_op_int("es_compensate_fallback", "L", L, ES_INT)), static_cast<int>(es_op_int("es_compensate_fallback", "H", H, ES_INT)), static_cast<int>(es_op_int("es_compensate_fallback", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_compensate_fallback(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& v_mean, const c10::optional<at::Tensor>& keep, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& flags, int64_t L, int64_t H, int64_t D) {}

static void op_es_dense_attention(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse2, int64_t L, int64_t H, int64_t D) {
  const Call es_op_call("es_dense_attention", {&q, &k, &v, &out, &lse2});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_dense_attention", es_dense_attention(static_cast<const void*>(es_op_data("es_dense_attention", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("es_dense_attention", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("es_dense_attention", "v", v, ES_HALF)), static_cast<void*>(es_op_data("es_dense_attention", "out", out, ES_OUT)), static_cast<float*>(es_op_data("es_dense_attention", "lse2", lse2, ES_F32)), static_cast<int>(es_op_int("es_dense_attention", "L", L, ES_INT)), static_cast<int>(es_op_int("es_dense_attention", "H", H, ES_INT)), static_cast<int>(es_op_int("es_dense_attention", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_dense_attention(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse2, int64_t L, int64_t H, int64_t D) {}

static void op_es_dense_attention_kv(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse2, int64_t Lq, int64_t Lk, int64_t H, int64_t D) {
  const Call es_op_call("es_dense_attention_kv", {&q, &k, &v, &out, &lse2});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_dense_attention_kv", es_dense_attention_kv(static_cast<const void*>(es_op_data("es_dense_attention_kv", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("es_dense_attention_kv", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("es_dense_attention_kv", "v", v, ES_HALF)), static_cast<void*>(es_op_data("es_dense_attention_kv", "out", out, ES_OUT)), static_cast<float*>(es_op_data("es_dense_attention_kv", "lse2", lse2, ES_F32)), static_cast<int>(es_op_int("es_dense_attention_kv", "Lq", Lq, ES_INT)), static_cast<int>(es_op_int("es_dense_attention_kv", "Lk", Lk, ES_INT)), static_cast<int>(es_op_int("es_dense_attention_kv", "H", H, ES_INT)), static_cast<int>(es_op_int("es_dense_attention_kv", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_dense_attention_kv(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse2, int64_t Lq, int64_t Lk, int64_t H, int64_t D) {}

static void op_es_dense_attention_ws(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse2, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes, int64_t Lq, int64_t Lk, int64_t H, int64_t D) {
  const Call es_op_call("es_dense_attention_ws", {&q, &k, &v, &out, &lse2, &workspace});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_dense_attention_ws", es_dense_attention_ws(static_cast<const void*>(es_op_data("es_dense_attention_ws", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("es_dense_attention_ws", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("es_dense_attention_ws", "v", v, ES_HALF)), static_cast<void*>(es_op_data("es_dense_attention_ws", "out", out, ES_OUT)), static_cast<float*>(es_op_data("es_dense_attention_ws", "lse2", lse2, ES_F32)), static_cast<void*>(es_op_data("es_dense_attention_ws", "workspace", workspace, ES_ANY)), static_cast<size_t>(es_op_int("es_dense_attention_ws", "workspace_bytes", workspace_bytes, ES_SIZE)), static_cast<int>(es_op_int("es_dense_attention_ws", "Lq", Lq, ES_INT)), static_cast<int>(es_op_int("es_dense_attention_ws", "Lk", Lk, ES_INT)), static_cast<int>(es_op_int("es_dense_attention_ws", "H", H, ES_INT)), static_cast<int>(es_op_int("es_dense_attention_ws", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_dense_attention_ws(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse2, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes, int64_t Lq, int64_t Lk, int64_t H, int64_t D) {}

static void op_es_block_means(const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& v_mean, int64_t L, int64_t H, int64_t D) {
  const Call es_op_call("es_block_means", {&k, &v, &k_mean, &v_mean});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_block_means", es_block_means(static_cast<const void*>(es_op_data("es_block_means", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("es_block_means", "v", v, ES_HALF)), static_cast<void*>(es_op_data("es_block_means", "k_mean", k_mean, ES_OUT)), static_cast<void*>(es_op_data("es_block_means", "v_mean", v_mean, ES_OUT)), static_cast<int>(es_op_int("es_block_means", "L", L, ES_INT)), static_cast<int>(es_op_int("es_block_means", "H", H, ES_INT)), static_cast<int>(es_op_int("es_block_means", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_block_means(const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& v_mean, int64_t L, int64_t H, int64_t D) {}

static void op_es_estimate_skipped(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& keep, const c10::optional<at::Tensor>& offset, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& mass, const c10::optional<at::Tensor>& scale_exact, const c10::optional<at::Tensor>& scale_skip, int64_t L, int64_t H, int64_t D) {
  const Call es_op_call("es_estimate_skipped", {&q, &k_mean, &keep, &offset, &lse, &mass, &scale_exact, &scale_skip});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_estimate_skipped", es_estimate_skipped(static_cast<const void*>(es_op_data("es_estimate_skipped", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("es_estimate_skipped", "k_mean", k_mean, ES_HALF)), static_cast<const uint8_t*>(es_op_data("es_estimate_skipped", "keep", keep, ES_U8)), static_cast<const float*>(es_op_data("es_estimate_skipped", "offset", offset, ES_F32)), static_cast<const float*>(es_op_data("es_estimate_skipped", "lse", lse, ES_F32)), static_cast<float*>(es_op_data("es_estimate_skipped", "mass", mass, ES_F32)), static_cast<float*>(es_op_data("es_estimate_skipped", "scale_exact", scale_exact, ES_F32)), static_cast<float*>(es_op_data("es_estimate_skipped", "scale_skip", scale_skip, ES_F32)), static_cast<int>(es_op_int("es_estimate_skipped", "L", L, ES_INT)), static_cast<int>(es_op_int("es_estimate_skipped", "H", H, ES_INT)), static_cast<int>(es_op_int("es_estimate_skipped", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_estimate_skipped(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& keep, const c10::optional<at::Tensor>& offset, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& mass, const c10::optional<at::Tensor>& scale_exact, const c10::optional<at::Tensor>& scale_skip, int64_t L, int64_t H, int64_t D) {}

static void op_es_full_step_scales(const c10::optional<at::Tensor>& offset, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& scale_exact, const c10::optional<at::Tensor>& scale_skip, int64_t L, int64_t H) {
  const Call es_op_call("es_full_step_scales", {&offset, &lse, &scale_exact, &scale_skip});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_full_step_scales", es_full_step_scales(static_cast<const float*>(es_op_data("es_full_step_scales", "offset", offset, ES_F32)), static_cast<float*>(es_op_data("es_full_step_scales", "lse", lse, ES_F32)), static_cast<float*>(es_op_data("es_full_step_scales", "scale_exact", scale_exact, ES_F32)), static_cast<float*>(es_op_data("es_full_step_scales", "scale_skip", scale_skip, ES_F32)), static_cast<int>(es_op_int("es_full_step_scales", "L", L, ES_INT)), static_cast<int>(es_op_int("es_full_step_scales", "H", H, ES_INT)), es_op_stream));
}
static void meta_es_full_step_scales(const c10::optional<at::Tensor>& offset, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& scale_exact, const c10::optional<at::Tensor>& scale_skip, int64_t L, int64_t H) {}

static void op_es_select_blocks(const c10::optional<at::Tensor>& mass, const c10::optional<at::Tensor>& keep_prev, const c10::optional<at::Tensor>& scale_exact, const c10::optional<at::Tensor>& scale_skip, const c10::optional<at::Tensor>& keep, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& blocks, const c10::optional<at::Tensor>& flags, const c10::optional<at::Tensor>& skip_bits, int64_t nw, const c10::optional<at::Tensor>& refine, int64_t rw, int64_t k, int64_t r, int64_t L, int64_t H, int64_t sink) {
  const Call es_op_call("es_select_blocks", {&mass, &keep_prev, &scale_exact, &scale_skip, &keep, &counts, &blocks, &flags, &skip_bits, &refine});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_select_blocks", es_select_blocks(static_cast<const float*>(es_op_data("es_select_blocks", "mass", mass, ES_F32)), static_cast<const uint8_t*>(es_op_data("es_select_blocks", "keep_prev", keep_prev, ES_U8)), static_cast<const float*>(es_op_data("es_select_blocks", "scale_exact", scale_exact, ES_F32)), static_cast<const float*>(es_op_data("es_select_blocks", "scale_skip", scale_skip, ES_F32)), static_cast<uint8_t*>(es_op_data("es_select_blocks", "keep", keep, ES_U8)), static_cast<int*>(es_op_data("es_select_blocks", "counts", counts, ES_I32)), static_cast<int*>(es_op_data("es_select_blocks", "blocks", blocks, ES_I32)), static_cast<const int*>(es_op_data("es_select_blocks", "flags", flags, ES_I32)), static_cast<int*>(es_op_data("es_select_blocks", "skip_bits", skip_bits, ES_I32)), static_cast<int>(es_op_int("es_select_blocks", "nw", nw, ES_INT)), static_cast<int*>(es_op_data("es_select_blocks", "refine", refine, ES_I32)), static_cast<int>(es_op_int("es_select_blocks", "rw", rw, ES_INT)), static_cast<int>(es_op_int("es_select_blocks", "k", k, ES_INT)), static_cast<int>(es_op_int("es_select_blocks", "r", r, ES_INT)), static_cast<int>(es_op_int("es_select_blocks", "L", L, ES_INT)), static_cast<int>(es_op_int("es_select_blocks", "H", H, ES_INT)), static_cast<int>(es_op_int("es_select_blocks", "sink", sink, ES_INT)), es_op_stream));
}
static void meta_es_select_blocks(const c10::optional<at::Tensor>& mass, const c10::optional<at::Tensor>& keep_prev, const c10::optional<at::Tensor>& scale_exact, const c10::optional<at::Tensor>& scale_skip, const c10::optional<at::Tensor>& keep, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& blocks, const c10::optional<at::Tensor>& flags, const c10::optional<at::Tensor>& skip_bits, int64_t nw, const c10::optional<at::Tensor>& refine, int64_t rw, int64_t k, int64_t r, int64_t L, int64_t H, int64_t sink) {}

static void op_es_pack_plan(const c10::optional<at::Tensor>& keep, const c10::optional<at::Tensor>& exact_bits, int64_t nw, int64_t H, int64_t nq, int64_t nb) {
  const Call es_op_call("es_pack_plan", {&keep, &exact_bits});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_pack_plan", es_pack_plan(static_cast<const uint8_t*>(es_op_data("es_pack_plan", "keep", keep, ES_U8)), static_cast<int*>(es_op_data("es_pack_plan", "exact_bits", exact_bits, ES_I32)), static_cast<int>(es_op_int("es_pack_plan", "nw", nw, ES_INT)), static_cast<int>(es_op_int("es_pack_plan", "H", H, ES_INT)), static_cast<int>(es_op_int("es_pack_plan", "nq", nq, ES_INT)), static_cast<int>(es_op_int("es_pack_plan", "nb", nb, ES_INT)), es_op_stream));
}
static void meta_es_pack_plan(const c10::optional<at::Tensor>& keep, const c10::optional<at::Tensor>& exact_bits, int64_t nw, int64_t H, int64_t nq, int64_t nb) {}

static void op_es_rebuild_plan(const c10::optional<at::Tensor>& exact_bits, const c10::optional<at::Tensor>& skip_bits, int64_t nw, const c10::optional<at::Tensor>& keep, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& blocks, const c10::optional<at::Tensor>& refine, const c10::optional<at::Tensor>& refine_counts, int64_t rw, const c10::optional<at::Tensor>& means, const c10::optional<at::Tensor>& mean_counts, int64_t H, int64_t nq, int64_t nb) {
  const Call es_op_call("es_rebuild_plan", {&exact_bits, &skip_bits, &keep, &counts, &blocks, &refine, &refine_counts, &means, &mean_counts});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_rebuild_plan", es_rebuild_plan(static_cast<const int*>(es_op_data("es_rebuild_plan", "exact_bits", exact_bits, ES_I32)), static_cast<const int*>(es_op_data("es_rebuild_plan", "skip_bits", skip_bits, ES_I32)), static_cast<int>(es_op_int("es_rebuild_plan", "nw", nw, ES_INT)), static_cast<uint8_t*>(es_op_data("es_rebuild_plan", "keep", keep, ES_U8)), static_cast<int*>(es_op_data("es_rebuild_plan", "counts", counts, ES_I32)), static_cast<int*>(es_op_data("es_rebuild_plan", "blocks", blocks, ES_I32)), static_cast<int*>(es_op_data("es_rebuild_plan", "refine", refine, ES_I32)), static_cast<int*>(es_op_data("es_rebuild_plan", "refine_counts", refine_counts, ES_I32)), static_cast<int>(es_op_int("es_rebuild_plan", "rw", rw, ES_INT)), static_cast<int*>(es_op_data("es_rebuild_plan", "means", means, ES_I32)), static_cast<int*>(es_op_data("es_rebuild_plan", "mean_counts", mean_counts, ES_I32)), static_cast<int>(es_op_int("es_rebuild_plan", "H", H, ES_INT)), static_cast<int>(es_op_int("es_rebuild_plan", "nq", nq, ES_INT)), static_cast<int>(es_op_int("es_rebuild_plan", "nb", nb, ES_INT)), es_op_stream));
}
static void meta_es_rebuild_plan(const c10::optional<at::Tensor>& exact_bits, const c10::optional<at::Tensor>& skip_bits, int64_t nw, const c10::optional<at::Tensor>& keep, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& blocks, const c10::optional<at::Tensor>& refine, const c10::optional<at::Tensor>& refine_counts, int64_t rw, const c10::optional<at::Tensor>& means, const c10::optional<at::Tensor>& mean_counts, int64_t H, int64_t nq, int64_t nb) {}

static void op_es_representatives(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_rep, const c10::optional<at::Tensor>& v_rep, const c10::optional<at::Tensor>& log_counts, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& v_mean, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes, int64_t iters, int64_t L, int64_t H, int64_t D) {
  const Call es_op_call("es_representatives", {&q, &k, &v, &k_rep, &v_rep, &log_counts, &k_mean, &v_mean, &workspace});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_representatives", es_representatives(static_cast<const void*>(es_op_data("es_representatives", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("es_representatives", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("es_representatives", "v", v, ES_HALF)), static_cast<void*>(es_op_data("es_representatives", "k_rep", k_rep, ES_OUT)), static_cast<void*>(es_op_data("es_representatives", "v_rep", v_rep, ES_OUT)), static_cast<float*>(es_op_data("es_representatives", "log_counts", log_counts, ES_F32)), static_cast<void*>(es_op_data("es_representatives", "k_mean", k_mean, ES_OUT)), static_cast<void*>(es_op_data("es_representatives", "v_mean", v_mean, ES_OUT)), static_cast<void*>(es_op_data("es_representatives", "workspace", workspace, ES_ANY)), static_cast<size_t>(es_op_int("es_representatives", "workspace_bytes", workspace_bytes, ES_SIZE)), static_cast<int>(es_op_int("es_representatives", "iters", iters, ES_INT)), static_cast<int>(es_op_int("es_representatives", "L", L, ES_INT)), static_cast<int>(es_op_int("es_representatives", "H", H, ES_INT)), static_cast<int>(es_op_int("es_representatives", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_representatives(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_rep, const c10::optional<at::Tensor>& v_rep, const c10::optional<at::Tensor>& log_counts, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& v_mean, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes, int64_t iters, int64_t L, int64_t H, int64_t D) {}

static void op_es_representatives_noalloc(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_rep, const c10::optional<at::Tensor>& v_rep, const c10::optional<at::Tensor>& log_counts, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& v_mean, int64_t iters, int64_t L, int64_t H, int64_t D) {
  const Call es_op_call("es_representatives_noalloc", {&q, &k, &v, &k_rep, &v_rep, &log_counts, &k_mean, &v_mean});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("es_representatives_noalloc", es_representatives_noalloc(static_cast<const void*>(es_op_data("es_representatives_noalloc", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("es_representatives_noalloc", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("es_representatives_noalloc", "v", v, ES_HALF)), static_cast<void*>(es_op_data("es_representatives_noalloc", "k_rep", k_rep, ES_OUT)), static_cast<void*>(es_op_data("es_representatives_noalloc", "v_rep", v_rep, ES_OUT)), static_cast<float*>(es_op_data("es_representatives_noalloc", "log_counts", log_counts, ES_F32)), static_cast<void*>(es_op_data("es_representatives_noalloc", "k_mean", k_mean, ES_OUT)), static_cast<void*>(es_op_data("es_representatives_noalloc", "v_mean", v_mean, ES_OUT)), static_cast<int>(es_op_int("es_representatives_noalloc", "iters", iters, ES_INT)), static_cast<int>(es_op_int("es_representatives_noalloc", "L", L, ES_INT)), static_cast<int>(es_op_int("es_representatives_noalloc", "H", H, ES_INT)), static_cast<int>(es_op_int("es_representatives_noalloc", "D", D, ES_INT)), es_op_stream));
}
static void meta_es_representatives_noalloc(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_rep, const c10::optional<at::Tensor>& v_rep, const c10::optional<at::Tensor>& log_counts, const c10::optional<at::Tensor>& k_mean, const c10::optional<at::Tensor>& v_mean, int64_t iters, int64_t L, int64_t H, int64_t D) {}

static void op_vsa_pool(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& vr, const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, const c10::optional<at::Tensor>& vc, int64_t BH, int64_t L, int64_t D, int64_t R) {
  const Call es_op_call("vsa_pool", {&q, &k, &v, &blk_cnt, &qr, &kr, &vr, &qc, &kc, &vc});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_pool", vsa_pool(static_cast<const void*>(es_op_data("vsa_pool", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_pool", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_pool", "v", v, ES_HALF)), static_cast<const int*>(es_op_data("vsa_pool", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_pool", "qr", qr, ES_OUT)), static_cast<void*>(es_op_data("vsa_pool", "kr", kr, ES_OUT)), static_cast<void*>(es_op_data("vsa_pool", "vr", vr, ES_OUT)), static_cast<void*>(es_op_data("vsa_pool", "qc", qc, ES_OUT)), static_cast<void*>(es_op_data("vsa_pool", "kc", kc, ES_OUT)), static_cast<void*>(es_op_data("vsa_pool", "vc", vc, ES_OUT)), static_cast<int>(es_op_int("vsa_pool", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_pool", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_pool", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_pool", "R", R, ES_INT)), es_op_stream));
}
static void meta_vsa_pool(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& vr, const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, const c10::optional<at::Tensor>& vc, int64_t BH, int64_t L, int64_t D, int64_t R) {}

static void op_vsa_fuse_fwd(const c10::optional<at::Tensor>& of, const c10::optional<at::Tensor>& oc, const c10::optional<at::Tensor>& gate, const c10::optional<at::Tensor>& o, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D, int64_t NBc_pad, int64_t gate_mode, int64_t gate_act) {
  const Call es_op_call("vsa_fuse_fwd", {&of, &oc, &gate, &o, &blk_cnt});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_fuse_fwd", vsa_fuse_fwd(static_cast<const void*>(es_op_data("vsa_fuse_fwd", "of", of, ES_HALF)), static_cast<const void*>(es_op_data("vsa_fuse_fwd", "oc", oc, ES_HALF)), static_cast<const void*>(es_op_data("vsa_fuse_fwd", "gate", gate, ES_HALF)), static_cast<void*>(es_op_data("vsa_fuse_fwd", "o", o, ES_OUT)), static_cast<const int*>(es_op_data("vsa_fuse_fwd", "blk_cnt", blk_cnt, ES_I32)), static_cast<int>(es_op_int("vsa_fuse_fwd", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_fwd", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_fwd", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_fwd", "NBc_pad", NBc_pad, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_fwd", "gate_mode", gate_mode, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_fwd", "gate_act", gate_act, ES_INT)), es_op_stream));
}
static void meta_vsa_fuse_fwd(const c10::optional<at::Tensor>& of, const c10::optional<at::Tensor>& oc, const c10::optional<at::Tensor>& gate, const c10::optional<at::Tensor>& o, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D, int64_t NBc_pad, int64_t gate_mode, int64_t gate_act) {}

static void op_vsa_fuse_bwd(const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& of, const c10::optional<at::Tensor>& oc, const c10::optional<at::Tensor>& gate, const c10::optional<at::Tensor>& dout_f, const c10::optional<at::Tensor>& delta_f, const c10::optional<at::Tensor>& dout_c, const c10::optional<at::Tensor>& delta_c, const c10::optional<at::Tensor>& dgate, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D, int64_t NBc_pad, int64_t gate_mode, int64_t gate_act) {
  const Call es_op_call("vsa_fuse_bwd", {&dout, &of, &oc, &gate, &dout_f, &delta_f, &dout_c, &delta_c, &dgate, &blk_cnt});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_fuse_bwd", vsa_fuse_bwd(static_cast<const void*>(es_op_data("vsa_fuse_bwd", "dout", dout, ES_HALF)), static_cast<const void*>(es_op_data("vsa_fuse_bwd", "of", of, ES_HALF)), static_cast<const void*>(es_op_data("vsa_fuse_bwd", "oc", oc, ES_HALF)), static_cast<const void*>(es_op_data("vsa_fuse_bwd", "gate", gate, ES_HALF)), static_cast<void*>(es_op_data("vsa_fuse_bwd", "dout_f", dout_f, ES_OUT)), static_cast<float*>(es_op_data("vsa_fuse_bwd", "delta_f", delta_f, ES_F32)), static_cast<void*>(es_op_data("vsa_fuse_bwd", "dout_c", dout_c, ES_OUT)), static_cast<float*>(es_op_data("vsa_fuse_bwd", "delta_c", delta_c, ES_F32)), static_cast<void*>(es_op_data("vsa_fuse_bwd", "dgate", dgate, ES_OUT)), static_cast<const int*>(es_op_data("vsa_fuse_bwd", "blk_cnt", blk_cnt, ES_I32)), static_cast<int>(es_op_int("vsa_fuse_bwd", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_bwd", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_bwd", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_bwd", "NBc_pad", NBc_pad, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_bwd", "gate_mode", gate_mode, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_bwd", "gate_act", gate_act, ES_INT)), es_op_stream));
}
static void meta_vsa_fuse_bwd(const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& of, const c10::optional<at::Tensor>& oc, const c10::optional<at::Tensor>& gate, const c10::optional<at::Tensor>& dout_f, const c10::optional<at::Tensor>& delta_f, const c10::optional<at::Tensor>& dout_c, const c10::optional<at::Tensor>& delta_c, const c10::optional<at::Tensor>& dgate, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D, int64_t NBc_pad, int64_t gate_mode, int64_t gate_act) {}

static void op_vsa_finalize(const c10::optional<at::Tensor>& acc, const c10::optional<at::Tensor>& add, int64_t add_nb, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_finalize", {&acc, &add, &out, &blk_cnt});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_finalize", vsa_finalize(static_cast<const float*>(es_op_data("vsa_finalize", "acc", acc, ES_F32)), static_cast<const float*>(es_op_data("vsa_finalize", "add", add, ES_F32)), static_cast<int>(es_op_int("vsa_finalize", "add_nb", add_nb, ES_INT)), static_cast<void*>(es_op_data("vsa_finalize", "out", out, ES_OUT)), static_cast<const int*>(es_op_data("vsa_finalize", "blk_cnt", blk_cnt, ES_I32)), static_cast<int>(es_op_int("vsa_finalize", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_finalize", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_finalize", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_finalize(const c10::optional<at::Tensor>& acc, const c10::optional<at::Tensor>& add, int64_t add_nb, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_fwd(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& row_ptr, const c10::optional<at::Tensor>& col_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_fwd", {&q, &k, &v, &row_ptr, &col_idx, &blk_cnt, &out, &lse});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_fwd", vsa_attn_fwd(static_cast<const void*>(es_op_data("vsa_attn_fwd", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_fwd", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_fwd", "v", v, ES_HALF)), static_cast<const int*>(es_op_data("vsa_attn_fwd", "row_ptr", row_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_fwd", "col_idx", col_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_fwd", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_attn_fwd", "out", out, ES_OUT)), static_cast<float*>(es_op_data("vsa_attn_fwd", "lse", lse, ES_F32)), static_cast<int>(es_op_int("vsa_attn_fwd", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_fwd", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_fwd", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_fwd(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& row_ptr, const c10::optional<at::Tensor>& col_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_fwd_tasks(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& col_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& part_o, const c10::optional<at::Tensor>& part_lse, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_fwd_tasks", {&q, &k, &v, &col_idx, &blk_cnt, &tasks, &info, &out, &lse, &part_o, &part_lse});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_fwd_tasks", vsa_attn_fwd_tasks(static_cast<const void*>(es_op_data("vsa_attn_fwd_tasks", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_fwd_tasks", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_fwd_tasks", "v", v, ES_HALF)), static_cast<const int*>(es_op_data("vsa_attn_fwd_tasks", "col_idx", col_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_fwd_tasks", "blk_cnt", blk_cnt, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_fwd_tasks", "tasks", tasks, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_fwd_tasks", "info", info, ES_I32)), static_cast<int>(es_op_int("vsa_attn_fwd_tasks", "max_tasks", max_tasks, ES_INT)), static_cast<void*>(es_op_data("vsa_attn_fwd_tasks", "out", out, ES_OUT)), static_cast<float*>(es_op_data("vsa_attn_fwd_tasks", "lse", lse, ES_F32)), static_cast<float*>(es_op_data("vsa_attn_fwd_tasks", "part_o", part_o, ES_F32)), static_cast<float*>(es_op_data("vsa_attn_fwd_tasks", "part_lse", part_lse, ES_F32)), static_cast<int>(es_op_int("vsa_attn_fwd_tasks", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_fwd_tasks", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_fwd_tasks", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_fwd_tasks(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& col_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& part_o, const c10::optional<at::Tensor>& part_lse, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_bwd_kv(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dk, const c10::optional<at::Tensor>& add_dv, int64_t add_nb, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, int64_t out_fp32, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_bwd_kv", {&q, &k, &v, &dout, &lse, &delta, &k2q_ptr, &k2q_idx, &blk_cnt, &add_dk, &add_dv, &dk, &dv});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_bwd_kv", vsa_attn_bwd_kv(static_cast<const void*>(es_op_data("vsa_attn_bwd_kv", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv", "dout", dout, ES_HALF)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv", "delta", delta, ES_F32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv", "k2q_ptr", k2q_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv", "k2q_idx", k2q_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv", "blk_cnt", blk_cnt, ES_I32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv", "add_dk", add_dk, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv", "add_dv", add_dv, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_kv", "add_nb", add_nb, ES_INT)), static_cast<void*>(es_op_data("vsa_attn_bwd_kv", "dk", dk, ES_OUT)), static_cast<void*>(es_op_data("vsa_attn_bwd_kv", "dv", dv, ES_OUT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv", "out_fp32", out_fp32, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_bwd_kv(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dk, const c10::optional<at::Tensor>& add_dv, int64_t add_nb, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, int64_t out_fp32, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_bwd_kv_tasks(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& add_dk, const c10::optional<at::Tensor>& add_dv, int64_t add_nb, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, const c10::optional<at::Tensor>& part_dk, const c10::optional<at::Tensor>& part_dv, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_bwd_kv_tasks", {&q, &k, &v, &dout, &lse, &delta, &k2q_idx, &blk_cnt, &tasks, &info, &add_dk, &add_dv, &dk, &dv, &part_dk, &part_dv});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_bwd_kv_tasks", vsa_attn_bwd_kv_tasks(static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_tasks", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_tasks", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_tasks", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_tasks", "dout", dout, ES_HALF)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_tasks", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_tasks", "delta", delta, ES_F32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_tasks", "k2q_idx", k2q_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_tasks", "blk_cnt", blk_cnt, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_tasks", "tasks", tasks, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_tasks", "info", info, ES_I32)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_tasks", "max_tasks", max_tasks, ES_INT)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_tasks", "add_dk", add_dk, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_tasks", "add_dv", add_dv, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_tasks", "add_nb", add_nb, ES_INT)), static_cast<void*>(es_op_data("vsa_attn_bwd_kv_tasks", "dk", dk, ES_OUT)), static_cast<void*>(es_op_data("vsa_attn_bwd_kv_tasks", "dv", dv, ES_OUT)), static_cast<float*>(es_op_data("vsa_attn_bwd_kv_tasks", "part_dk", part_dk, ES_F32)), static_cast<float*>(es_op_data("vsa_attn_bwd_kv_tasks", "part_dv", part_dv, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_tasks", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_tasks", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_tasks", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_bwd_kv_tasks(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& add_dk, const c10::optional<at::Tensor>& add_dv, int64_t add_nb, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, const c10::optional<at::Tensor>& part_dk, const c10::optional<at::Tensor>& part_dv, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_bwd_q(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq, const c10::optional<at::Tensor>& dq_acc, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_bwd_q", {&q, &k, &v, &dout, &lse, &delta, &q2k_ptr, &q2k_idx, &blk_cnt, &add_dq, &dq, &dq_acc});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_bwd_q", vsa_attn_bwd_q(static_cast<const void*>(es_op_data("vsa_attn_bwd_q", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q", "dout", dout, ES_HALF)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q", "delta", delta, ES_F32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q", "q2k_idx", q2k_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q", "blk_cnt", blk_cnt, ES_I32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q", "add_dq", add_dq, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_q", "add_nb", add_nb, ES_INT)), static_cast<void*>(es_op_data("vsa_attn_bwd_q", "dq", dq, ES_OUT)), static_cast<float*>(es_op_data("vsa_attn_bwd_q", "dq_acc", dq_acc, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_q", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_q", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_q", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_bwd_q(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq, const c10::optional<at::Tensor>& dq_acc, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_bwd_q_tasks(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq, const c10::optional<at::Tensor>& part_dq, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_bwd_q_tasks", {&q, &k, &v, &dout, &lse, &delta, &q2k_idx, &blk_cnt, &tasks, &info, &add_dq, &dq, &part_dq});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_bwd_q_tasks", vsa_attn_bwd_q_tasks(static_cast<const void*>(es_op_data("vsa_attn_bwd_q_tasks", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q_tasks", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q_tasks", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q_tasks", "dout", dout, ES_HALF)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q_tasks", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q_tasks", "delta", delta, ES_F32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_tasks", "q2k_idx", q2k_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_tasks", "blk_cnt", blk_cnt, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_tasks", "tasks", tasks, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_tasks", "info", info, ES_I32)), static_cast<int>(es_op_int("vsa_attn_bwd_q_tasks", "max_tasks", max_tasks, ES_INT)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q_tasks", "add_dq", add_dq, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_q_tasks", "add_nb", add_nb, ES_INT)), static_cast<void*>(es_op_data("vsa_attn_bwd_q_tasks", "dq", dq, ES_OUT)), static_cast<float*>(es_op_data("vsa_attn_bwd_q_tasks", "part_dq", part_dq, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_q_tasks", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_q_tasks", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_q_tasks", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_bwd_q_tasks(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq, const c10::optional<at::Tensor>& part_dq, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_block_scores(const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, const c10::optional<at::Tensor>& scores, int64_t NB, int64_t NBc_pad, int64_t bh0, int64_t bh_count, int64_t D) {
  const Call es_op_call("vsa_block_scores", {&qc, &kc, &scores});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_block_scores", vsa_block_scores(static_cast<const void*>(es_op_data("vsa_block_scores", "qc", qc, ES_HALF)), static_cast<const void*>(es_op_data("vsa_block_scores", "kc", kc, ES_HALF)), static_cast<void*>(es_op_data("vsa_block_scores", "scores", scores, ES_OUT)), static_cast<int>(es_op_int("vsa_block_scores", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_block_scores", "NBc_pad", NBc_pad, ES_INT)), static_cast<int>(es_op_int("vsa_block_scores", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_block_scores", "bh_count", bh_count, ES_INT)), static_cast<int>(es_op_int("vsa_block_scores", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_block_scores(const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, const c10::optional<at::Tensor>& scores, int64_t NB, int64_t NBc_pad, int64_t bh0, int64_t bh_count, int64_t D) {}

static void op_vsa_route_rows(const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, int64_t NB, int64_t NBc_pad, int64_t bh0, int64_t bh_count, int64_t K, int64_t D, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {
  const Call es_op_call("vsa_route_rows", {&qc, &kc, &q2k_ptr, &q2k_idx, &k2q_ptr, &k2q_idx, &workspace});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_route_rows", vsa_route_rows(static_cast<const void*>(es_op_data("vsa_route_rows", "qc", qc, ES_HALF)), static_cast<const void*>(es_op_data("vsa_route_rows", "kc", kc, ES_HALF)), static_cast<int>(es_op_int("vsa_route_rows", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_route_rows", "NBc_pad", NBc_pad, ES_INT)), static_cast<int>(es_op_int("vsa_route_rows", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_route_rows", "bh_count", bh_count, ES_INT)), static_cast<int>(es_op_int("vsa_route_rows", "K", K, ES_INT)), static_cast<int>(es_op_int("vsa_route_rows", "D", D, ES_INT)), static_cast<int*>(es_op_data("vsa_route_rows", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_route_rows", "q2k_idx", q2k_idx, ES_I32)), static_cast<int*>(es_op_data("vsa_route_rows", "k2q_ptr", k2q_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_route_rows", "k2q_idx", k2q_idx, ES_I32)), static_cast<void*>(es_op_data("vsa_route_rows", "workspace", workspace, ES_ANY)), static_cast<size_t>(es_op_int("vsa_route_rows", "workspace_bytes", workspace_bytes, ES_SIZE)), es_op_stream));
}
static void meta_vsa_route_rows(const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, int64_t NB, int64_t NBc_pad, int64_t bh0, int64_t bh_count, int64_t K, int64_t D, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {}

static void op_vsa_row_topk(const c10::optional<at::Tensor>& scores, int64_t NB, int64_t bh0, int64_t bh_count, int64_t K, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {
  const Call es_op_call("vsa_row_topk", {&scores, &q2k_ptr, &q2k_idx, &k2q_ptr, &k2q_idx, &workspace});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_row_topk", vsa_row_topk(static_cast<const void*>(es_op_data("vsa_row_topk", "scores", scores, ES_HALF)), static_cast<int>(es_op_int("vsa_row_topk", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_row_topk", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_row_topk", "bh_count", bh_count, ES_INT)), static_cast<int>(es_op_int("vsa_row_topk", "K", K, ES_INT)), static_cast<int*>(es_op_data("vsa_row_topk", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_row_topk", "q2k_idx", q2k_idx, ES_I32)), static_cast<int*>(es_op_data("vsa_row_topk", "k2q_ptr", k2q_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_row_topk", "k2q_idx", k2q_idx, ES_I32)), static_cast<void*>(es_op_data("vsa_row_topk", "workspace", workspace, ES_ANY)), static_cast<size_t>(es_op_int("vsa_row_topk", "workspace_bytes", workspace_bytes, ES_SIZE)), es_op_stream));
}
static void meta_vsa_row_topk(const c10::optional<at::Tensor>& scores, int64_t NB, int64_t bh0, int64_t bh_count, int64_t K, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {}

static void op_vsa_router_lse(const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& lse2, int64_t NB, int64_t R, int64_t BH, int64_t D) {
  const Call es_op_call("vsa_router_lse", {&qr, &kr, &blk_cnt, &lse2});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_router_lse", vsa_router_lse(static_cast<const void*>(es_op_data("vsa_router_lse", "qr", qr, ES_HALF)), static_cast<const void*>(es_op_data("vsa_router_lse", "kr", kr, ES_HALF)), static_cast<const int*>(es_op_data("vsa_router_lse", "blk_cnt", blk_cnt, ES_I32)), static_cast<float*>(es_op_data("vsa_router_lse", "lse2", lse2, ES_F32)), static_cast<int>(es_op_int("vsa_router_lse", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_router_lse", "R", R, ES_INT)), static_cast<int>(es_op_int("vsa_router_lse", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_router_lse", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_router_lse(const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& lse2, int64_t NB, int64_t R, int64_t BH, int64_t D) {}

static void op_vsa_router_scores(const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& lse2, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& scores, int64_t NB, int64_t R, int64_t row_norm, int64_t bh0, int64_t bh_count, int64_t D) {
  const Call es_op_call("vsa_router_scores", {&qr, &kr, &lse2, &blk_cnt, &scores});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_router_scores", vsa_router_scores(static_cast<const void*>(es_op_data("vsa_router_scores", "qr", qr, ES_HALF)), static_cast<const void*>(es_op_data("vsa_router_scores", "kr", kr, ES_HALF)), static_cast<const float*>(es_op_data("vsa_router_scores", "lse2", lse2, ES_F32)), static_cast<const int*>(es_op_data("vsa_router_scores", "blk_cnt", blk_cnt, ES_I32)), static_cast<float*>(es_op_data("vsa_router_scores", "scores", scores, ES_F32)), static_cast<int>(es_op_int("vsa_router_scores", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_router_scores", "R", R, ES_INT)), static_cast<int>(es_op_int("vsa_router_scores", "row_norm", row_norm, ES_INT)), static_cast<int>(es_op_int("vsa_router_scores", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_router_scores", "bh_count", bh_count, ES_INT)), static_cast<int>(es_op_int("vsa_router_scores", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_router_scores(const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& lse2, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& scores, int64_t NB, int64_t R, int64_t row_norm, int64_t bh0, int64_t bh_count, int64_t D) {}

static void op_vsa_global_topk(const c10::optional<at::Tensor>& scores, int64_t NB, int64_t bh0, int64_t bh_count, int64_t budget, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& bits_out, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {
  const Call es_op_call("vsa_global_topk", {&scores, &q2k_ptr, &q2k_idx, &k2q_ptr, &k2q_idx, &bits_out, &workspace});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_global_topk", vsa_global_topk(static_cast<const float*>(es_op_data("vsa_global_topk", "scores", scores, ES_F32)), static_cast<int>(es_op_int("vsa_global_topk", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_global_topk", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_global_topk", "bh_count", bh_count, ES_INT)), static_cast<long long>(es_op_int("vsa_global_topk", "budget", budget, ES_LL)), static_cast<int*>(es_op_data("vsa_global_topk", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_global_topk", "q2k_idx", q2k_idx, ES_I32)), static_cast<int*>(es_op_data("vsa_global_topk", "k2q_ptr", k2q_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_global_topk", "k2q_idx", k2q_idx, ES_I32)), static_cast<unsigned*>(es_op_data("vsa_global_topk", "bits_out", bits_out, ES_I32)), static_cast<void*>(es_op_data("vsa_global_topk", "workspace", workspace, ES_ANY)), static_cast<size_t>(es_op_int("vsa_global_topk", "workspace_bytes", workspace_bytes, ES_SIZE)), es_op_stream));
}
static void meta_vsa_global_topk(const c10::optional<at::Tensor>& scores, int64_t NB, int64_t bh0, int64_t bh_count, int64_t budget, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& bits_out, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {}

static void op_vsa_csr_transpose(const c10::optional<at::Tensor>& ptr, const c10::optional<at::Tensor>& idx, int64_t NB, int64_t bh0, int64_t bh_count, const c10::optional<at::Tensor>& out_ptr, const c10::optional<at::Tensor>& out_idx, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {
  const Call es_op_call("vsa_csr_transpose", {&ptr, &idx, &out_ptr, &out_idx, &workspace});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_csr_transpose", vsa_csr_transpose(static_cast<const int*>(es_op_data("vsa_csr_transpose", "ptr", ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_csr_transpose", "idx", idx, ES_I32)), static_cast<int>(es_op_int("vsa_csr_transpose", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_csr_transpose", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_csr_transpose", "bh_count", bh_count, ES_INT)), static_cast<int*>(es_op_data("vsa_csr_transpose", "out_ptr", out_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_csr_transpose", "out_idx", out_idx, ES_I32)), static_cast<void*>(es_op_data("vsa_csr_transpose", "workspace", workspace, ES_ANY)), static_cast<size_t>(es_op_int("vsa_csr_transpose", "workspace_bytes", workspace_bytes, ES_SIZE)), es_op_stream));
}
static void meta_vsa_csr_transpose(const c10::optional<at::Tensor>& ptr, const c10::optional<at::Tensor>& idx, int64_t NB, int64_t bh0, int64_t bh_count, const c10::optional<at::Tensor>& out_ptr, const c10::optional<at::Tensor>& out_idx, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {}

static void op_vsa_dense_lists(int64_t NB, int64_t BH, const c10::optional<at::Tensor>& cnt, const c10::optional<at::Tensor>& ptr, const c10::optional<at::Tensor>& idx) {
  const Call es_op_call("vsa_dense_lists", {&cnt, &ptr, &idx});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_dense_lists", vsa_dense_lists(static_cast<int>(es_op_int("vsa_dense_lists", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_dense_lists", "BH", BH, ES_INT)), static_cast<int*>(es_op_data("vsa_dense_lists", "cnt", cnt, ES_I32)), static_cast<int*>(es_op_data("vsa_dense_lists", "ptr", ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_dense_lists", "idx", idx, ES_I32)), es_op_stream));
}
static void meta_vsa_dense_lists(int64_t NB, int64_t BH, const c10::optional<at::Tensor>& cnt, const c10::optional<at::Tensor>& ptr, const c10::optional<at::Tensor>& idx) {}

static void op_vsa_split_plan(const c10::optional<at::Tensor>& ptr, int64_t BH, int64_t NB, int64_t chunk, int64_t max_slots, int64_t min_len, double rel_mean, double tail_frac, int64_t resident, int64_t budget, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& merges, const c10::optional<at::Tensor>& info) {
  const Call es_op_call("vsa_split_plan", {&ptr, &tasks, &merges, &info});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_split_plan", vsa_split_plan(static_cast<const int*>(es_op_data("vsa_split_plan", "ptr", ptr, ES_I32)), static_cast<int>(es_op_int("vsa_split_plan", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_split_plan", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_split_plan", "chunk", chunk, ES_INT)), static_cast<int>(es_op_int("vsa_split_plan", "max_slots", max_slots, ES_INT)), static_cast<int>(es_op_int("vsa_split_plan", "min_len", min_len, ES_INT)), static_cast<double>(rel_mean), static_cast<double>(tail_frac), static_cast<int>(es_op_int("vsa_split_plan", "resident", resident, ES_INT)), static_cast<int>(es_op_int("vsa_split_plan", "budget", budget, ES_INT)), static_cast<int*>(es_op_data("vsa_split_plan", "tasks", tasks, ES_I32)), static_cast<int*>(es_op_data("vsa_split_plan", "merges", merges, ES_I32)), static_cast<int*>(es_op_data("vsa_split_plan", "info", info, ES_I32)), es_op_stream));
}
static void meta_vsa_split_plan(const c10::optional<at::Tensor>& ptr, int64_t BH, int64_t NB, int64_t chunk, int64_t max_slots, int64_t min_len, double rel_mean, double tail_frac, int64_t resident, int64_t budget, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& merges, const c10::optional<at::Tensor>& info) {}

static void op_vsa_split_merge_fwd(const c10::optional<at::Tensor>& part_o, const c10::optional<at::Tensor>& part_lse, const c10::optional<at::Tensor>& merges, const c10::optional<at::Tensor>& info, int64_t max_merges, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& o, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D, int64_t mask_rows) {
  const Call es_op_call("vsa_split_merge_fwd", {&part_o, &part_lse, &merges, &info, &blk_cnt, &o, &lse});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_split_merge_fwd", vsa_split_merge_fwd(static_cast<const float*>(es_op_data("vsa_split_merge_fwd", "part_o", part_o, ES_F32)), static_cast<const float*>(es_op_data("vsa_split_merge_fwd", "part_lse", part_lse, ES_F32)), static_cast<const int*>(es_op_data("vsa_split_merge_fwd", "merges", merges, ES_I32)), static_cast<const int*>(es_op_data("vsa_split_merge_fwd", "info", info, ES_I32)), static_cast<int>(es_op_int("vsa_split_merge_fwd", "max_merges", max_merges, ES_INT)), static_cast<const int*>(es_op_data("vsa_split_merge_fwd", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_split_merge_fwd", "o", o, ES_OUT)), static_cast<float*>(es_op_data("vsa_split_merge_fwd", "lse", lse, ES_F32)), static_cast<int>(es_op_int("vsa_split_merge_fwd", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_split_merge_fwd", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_split_merge_fwd", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_split_merge_fwd", "mask_rows", mask_rows, ES_INT)), es_op_stream));
}
static void meta_vsa_split_merge_fwd(const c10::optional<at::Tensor>& part_o, const c10::optional<at::Tensor>& part_lse, const c10::optional<at::Tensor>& merges, const c10::optional<at::Tensor>& info, int64_t max_merges, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& o, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D, int64_t mask_rows) {}

static void op_vsa_split_merge_sum(const c10::optional<at::Tensor>& part, const c10::optional<at::Tensor>& merges, const c10::optional<at::Tensor>& info, int64_t max_merges, const c10::optional<at::Tensor>& add, int64_t add_nb, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& out_f32, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_split_merge_sum", {&part, &merges, &info, &add, &blk_cnt, &out, &out_f32});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_split_merge_sum", vsa_split_merge_sum(static_cast<const float*>(es_op_data("vsa_split_merge_sum", "part", part, ES_F32)), static_cast<const int*>(es_op_data("vsa_split_merge_sum", "merges", merges, ES_I32)), static_cast<const int*>(es_op_data("vsa_split_merge_sum", "info", info, ES_I32)), static_cast<int>(es_op_int("vsa_split_merge_sum", "max_merges", max_merges, ES_INT)), static_cast<const float*>(es_op_data("vsa_split_merge_sum", "add", add, ES_F32)), static_cast<int>(es_op_int("vsa_split_merge_sum", "add_nb", add_nb, ES_INT)), static_cast<const int*>(es_op_data("vsa_split_merge_sum", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_split_merge_sum", "out", out, ES_OUT)), static_cast<float*>(es_op_data("vsa_split_merge_sum", "out_f32", out_f32, ES_F32)), static_cast<int>(es_op_int("vsa_split_merge_sum", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_split_merge_sum", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_split_merge_sum", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_split_merge_sum(const c10::optional<at::Tensor>& part, const c10::optional<at::Tensor>& merges, const c10::optional<at::Tensor>& info, int64_t max_merges, const c10::optional<at::Tensor>& add, int64_t add_nb, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& out_f32, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_rep_build(const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, int64_t BH, int64_t L, int64_t D, int64_t RM) {
  const Call es_op_call("vsa_rep_build", {&k, &v, &blk_cnt, &k_mid, &v_mid, &lc_mid, &k_tail, &v_tail, &lc_tail});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_build", vsa_rep_build(static_cast<const void*>(es_op_data("vsa_rep_build", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_build", "v", v, ES_HALF)), static_cast<const int*>(es_op_data("vsa_rep_build", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_rep_build", "k_mid", k_mid, ES_OUT)), static_cast<void*>(es_op_data("vsa_rep_build", "v_mid", v_mid, ES_OUT)), static_cast<float*>(es_op_data("vsa_rep_build", "lc_mid", lc_mid, ES_F32)), static_cast<void*>(es_op_data("vsa_rep_build", "k_tail", k_tail, ES_OUT)), static_cast<void*>(es_op_data("vsa_rep_build", "v_tail", v_tail, ES_OUT)), static_cast<float*>(es_op_data("vsa_rep_build", "lc_tail", lc_tail, ES_F32)), static_cast<int>(es_op_int("vsa_rep_build", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build", "RM", RM, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_build(const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, int64_t BH, int64_t L, int64_t D, int64_t RM) {}

static void op_vsa_rep_build_kmeans(const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& labels, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t iters, int64_t seed) {
  const Call es_op_call("vsa_rep_build_kmeans", {&k, &v, &blk_cnt, &k_mid, &v_mid, &lc_mid, &counts, &labels});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_build_kmeans", vsa_rep_build_kmeans(static_cast<const void*>(es_op_data("vsa_rep_build_kmeans", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_build_kmeans", "v", v, ES_HALF)), static_cast<const int*>(es_op_data("vsa_rep_build_kmeans", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_rep_build_kmeans", "k_mid", k_mid, ES_OUT)), static_cast<void*>(es_op_data("vsa_rep_build_kmeans", "v_mid", v_mid, ES_OUT)), static_cast<float*>(es_op_data("vsa_rep_build_kmeans", "lc_mid", lc_mid, ES_F32)), static_cast<int*>(es_op_data("vsa_rep_build_kmeans", "counts", counts, ES_I32)), static_cast<uint8_t*>(es_op_data("vsa_rep_build_kmeans", "labels", labels, ES_U8)), static_cast<int>(es_op_int("vsa_rep_build_kmeans", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_kmeans", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_kmeans", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_kmeans", "RM", RM, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_kmeans", "iters", iters, ES_INT)), static_cast<unsigned>(es_op_int("vsa_rep_build_kmeans", "seed", seed, ES_UINT)), es_op_stream));
}
static void meta_vsa_rep_build_kmeans(const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& labels, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t iters, int64_t seed) {}

static void op_vsa_row_tiers(const c10::optional<at::Tensor>& scores, int64_t NB, int64_t bh0, int64_t bh_count, int64_t ka, int64_t kab, const c10::optional<at::Tensor>& a_ptr, const c10::optional<at::Tensor>& a_idx, const c10::optional<at::Tensor>& ab_ptr, const c10::optional<at::Tensor>& ab_idx, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab) {
  const Call es_op_call("vsa_row_tiers", {&scores, &a_ptr, &a_idx, &ab_ptr, &ab_idx, &bits_a, &bits_ab});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_row_tiers", vsa_row_tiers(static_cast<const float*>(es_op_data("vsa_row_tiers", "scores", scores, ES_F32)), static_cast<int>(es_op_int("vsa_row_tiers", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_row_tiers", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_row_tiers", "bh_count", bh_count, ES_INT)), static_cast<int>(es_op_int("vsa_row_tiers", "ka", ka, ES_INT)), static_cast<int>(es_op_int("vsa_row_tiers", "kab", kab, ES_INT)), static_cast<int*>(es_op_data("vsa_row_tiers", "a_ptr", a_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_row_tiers", "a_idx", a_idx, ES_I32)), static_cast<int*>(es_op_data("vsa_row_tiers", "ab_ptr", ab_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_row_tiers", "ab_idx", ab_idx, ES_I32)), static_cast<unsigned*>(es_op_data("vsa_row_tiers", "bits_a", bits_a, ES_I32)), static_cast<unsigned*>(es_op_data("vsa_row_tiers", "bits_ab", bits_ab, ES_I32)), es_op_stream));
}
static void meta_vsa_row_tiers(const c10::optional<at::Tensor>& scores, int64_t NB, int64_t bh0, int64_t bh_count, int64_t ka, int64_t kab, const c10::optional<at::Tensor>& a_ptr, const c10::optional<at::Tensor>& a_idx, const c10::optional<at::Tensor>& ab_ptr, const c10::optional<at::Tensor>& ab_idx, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab) {}

static void op_vsa_rep_attn_fwd(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t phases) {
  const Call es_op_call("vsa_rep_attn_fwd", {&q, &k, &v, &k_mid, &v_mid, &lc_mid, &k_tail, &v_tail, &lc_tail, &q2k_ptr, &q2k_idx, &bits_a, &bits_ab, &blk_cnt, &out, &lse});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_attn_fwd", vsa_rep_attn_fwd(static_cast<const void*>(es_op_data("vsa_rep_attn_fwd", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd", "k_mid", k_mid, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd", "v_mid", v_mid, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_attn_fwd", "lc_mid", lc_mid, ES_F32)), static_cast<int>(es_op_int("vsa_rep_attn_fwd", "lc_mid_stride", lc_mid_stride, ES_INT)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd", "k_tail", k_tail, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd", "v_tail", v_tail, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_attn_fwd", "lc_tail", lc_tail, ES_F32)), static_cast<const int*>(es_op_data("vsa_rep_attn_fwd", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_rep_attn_fwd", "q2k_idx", q2k_idx, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_attn_fwd", "bits_a", bits_a, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_attn_fwd", "bits_ab", bits_ab, ES_I32)), static_cast<const int*>(es_op_data("vsa_rep_attn_fwd", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_rep_attn_fwd", "out", out, ES_OUT)), static_cast<float*>(es_op_data("vsa_rep_attn_fwd", "lse", lse, ES_F32)), static_cast<int>(es_op_int("vsa_rep_attn_fwd", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_fwd", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_fwd", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_fwd", "RM", RM, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_fwd", "phases", phases, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_attn_fwd(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t phases) {}

static void op_vsa_rep_attn_bwd_q(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq_acc, const c10::optional<at::Tensor>& dq, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t phases) {
  const Call es_op_call("vsa_rep_attn_bwd_q", {&q, &k, &v, &k_mid, &v_mid, &lc_mid, &k_tail, &v_tail, &lc_tail, &dout, &lse, &delta, &q2k_ptr, &q2k_idx, &bits_a, &bits_ab, &blk_cnt, &add_dq, &dq_acc, &dq});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_attn_bwd_q", vsa_rep_attn_bwd_q(static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q", "k_mid", k_mid, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q", "v_mid", v_mid, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q", "lc_mid", lc_mid, ES_F32)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q", "lc_mid_stride", lc_mid_stride, ES_INT)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q", "k_tail", k_tail, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q", "v_tail", v_tail, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q", "lc_tail", lc_tail, ES_F32)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q", "dout", dout, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q", "delta", delta, ES_F32)), static_cast<const int*>(es_op_data("vsa_rep_attn_bwd_q", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_rep_attn_bwd_q", "q2k_idx", q2k_idx, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_attn_bwd_q", "bits_a", bits_a, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_attn_bwd_q", "bits_ab", bits_ab, ES_I32)), static_cast<const int*>(es_op_data("vsa_rep_attn_bwd_q", "blk_cnt", blk_cnt, ES_I32)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q", "add_dq", add_dq, ES_F32)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q", "add_nb", add_nb, ES_INT)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q", "dq_acc", dq_acc, ES_F32)), static_cast<void*>(es_op_data("vsa_rep_attn_bwd_q", "dq", dq, ES_OUT)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q", "RM", RM, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q", "phases", phases, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_attn_bwd_q(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq_acc, const c10::optional<at::Tensor>& dq, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t phases) {}

static void op_vsa_rep_bwd_tables(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& k_tab, const c10::optional<at::Tensor>& v_tab, const c10::optional<at::Tensor>& lc, int64_t lc_stride, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& dk_tab, const c10::optional<at::Tensor>& dv_tab, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t tier) {
  const Call es_op_call("vsa_rep_bwd_tables", {&q, &dout, &k_tab, &v_tab, &lc, &lse, &delta, &bits_a, &bits_ab, &dk_tab, &dv_tab});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_bwd_tables", vsa_rep_bwd_tables(static_cast<const void*>(es_op_data("vsa_rep_bwd_tables", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_tables", "dout", dout, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_tables", "k_tab", k_tab, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_tables", "v_tab", v_tab, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_bwd_tables", "lc", lc, ES_F32)), static_cast<int>(es_op_int("vsa_rep_bwd_tables", "lc_stride", lc_stride, ES_INT)), static_cast<const float*>(es_op_data("vsa_rep_bwd_tables", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_bwd_tables", "delta", delta, ES_F32)), static_cast<const unsigned*>(es_op_data("vsa_rep_bwd_tables", "bits_a", bits_a, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_bwd_tables", "bits_ab", bits_ab, ES_I32)), static_cast<float*>(es_op_data("vsa_rep_bwd_tables", "dk_tab", dk_tab, ES_F32)), static_cast<float*>(es_op_data("vsa_rep_bwd_tables", "dv_tab", dv_tab, ES_F32)), static_cast<int>(es_op_int("vsa_rep_bwd_tables", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_tables", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_tables", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_tables", "RM", RM, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_tables", "tier", tier, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_bwd_tables(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& k_tab, const c10::optional<at::Tensor>& v_tab, const c10::optional<at::Tensor>& lc, int64_t lc_stride, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& dk_tab, const c10::optional<at::Tensor>& dv_tab, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t tier) {}

static void op_vsa_rep_bwd_both_tables(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& dk_mid, const c10::optional<at::Tensor>& dv_mid, const c10::optional<at::Tensor>& dk_tail, const c10::optional<at::Tensor>& dv_tail, int64_t BH, int64_t L, int64_t D, int64_t RM) {
  const Call es_op_call("vsa_rep_bwd_both_tables", {&q, &dout, &k_mid, &v_mid, &lc_mid, &k_tail, &v_tail, &lc_tail, &lse, &delta, &bits_a, &bits_ab, &dk_mid, &dv_mid, &dk_tail, &dv_tail});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_bwd_both_tables", vsa_rep_bwd_both_tables(static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables", "dout", dout, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables", "k_mid", k_mid, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables", "v_mid", v_mid, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_bwd_both_tables", "lc_mid", lc_mid, ES_F32)), static_cast<int>(es_op_int("vsa_rep_bwd_both_tables", "lc_mid_stride", lc_mid_stride, ES_INT)), static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables", "k_tail", k_tail, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables", "v_tail", v_tail, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_bwd_both_tables", "lc_tail", lc_tail, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_bwd_both_tables", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_bwd_both_tables", "delta", delta, ES_F32)), static_cast<const unsigned*>(es_op_data("vsa_rep_bwd_both_tables", "bits_a", bits_a, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_bwd_both_tables", "bits_ab", bits_ab, ES_I32)), static_cast<float*>(es_op_data("vsa_rep_bwd_both_tables", "dk_mid", dk_mid, ES_F32)), static_cast<float*>(es_op_data("vsa_rep_bwd_both_tables", "dv_mid", dv_mid, ES_F32)), static_cast<float*>(es_op_data("vsa_rep_bwd_both_tables", "dk_tail", dk_tail, ES_F32)), static_cast<float*>(es_op_data("vsa_rep_bwd_both_tables", "dv_tail", dv_tail, ES_F32)), static_cast<int>(es_op_int("vsa_rep_bwd_both_tables", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_both_tables", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_both_tables", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_both_tables", "RM", RM, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_bwd_both_tables(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& dk_mid, const c10::optional<at::Tensor>& dv_mid, const c10::optional<at::Tensor>& dk_tail, const c10::optional<at::Tensor>& dv_tail, int64_t BH, int64_t L, int64_t D, int64_t RM) {}

static void op_vsa_rep_unpool(const c10::optional<at::Tensor>& acc_k, const c10::optional<at::Tensor>& acc_v, const c10::optional<at::Tensor>& dk_mid, const c10::optional<at::Tensor>& dv_mid, const c10::optional<at::Tensor>& dk_tail, const c10::optional<at::Tensor>& dv_tail, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& labels, const c10::optional<at::Tensor>& mid_counts, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, int64_t BH, int64_t L, int64_t D, int64_t RM) {
  const Call es_op_call("vsa_rep_unpool", {&acc_k, &acc_v, &dk_mid, &dv_mid, &dk_tail, &dv_tail, &blk_cnt, &labels, &mid_counts, &dk, &dv});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_unpool", vsa_rep_unpool(static_cast<const float*>(es_op_data("vsa_rep_unpool", "acc_k", acc_k, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_unpool", "acc_v", acc_v, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_unpool", "dk_mid", dk_mid, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_unpool", "dv_mid", dv_mid, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_unpool", "dk_tail", dk_tail, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_unpool", "dv_tail", dv_tail, ES_F32)), static_cast<const int*>(es_op_data("vsa_rep_unpool", "blk_cnt", blk_cnt, ES_I32)), static_cast<const uint8_t*>(es_op_data("vsa_rep_unpool", "labels", labels, ES_U8)), static_cast<const int*>(es_op_data("vsa_rep_unpool", "mid_counts", mid_counts, ES_I32)), static_cast<void*>(es_op_data("vsa_rep_unpool", "dk", dk, ES_OUT)), static_cast<void*>(es_op_data("vsa_rep_unpool", "dv", dv, ES_OUT)), static_cast<int>(es_op_int("vsa_rep_unpool", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_unpool", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_unpool", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_unpool", "RM", RM, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_unpool(const c10::optional<at::Tensor>& acc_k, const c10::optional<at::Tensor>& acc_v, const c10::optional<at::Tensor>& dk_mid, const c10::optional<at::Tensor>& dv_mid, const c10::optional<at::Tensor>& dk_tail, const c10::optional<at::Tensor>& dv_tail, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& labels, const c10::optional<at::Tensor>& mid_counts, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, int64_t BH, int64_t L, int64_t D, int64_t RM) {}

static void op_vsa_row_dot(const c10::optional<at::Tensor>& x, const c10::optional<at::Tensor>& y, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_row_dot", {&x, &y, &blk_cnt, &out});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_row_dot", vsa_row_dot(static_cast<const void*>(es_op_data("vsa_row_dot", "x", x, ES_HALF)), static_cast<const void*>(es_op_data("vsa_row_dot", "y", y, ES_HALF)), static_cast<const int*>(es_op_data("vsa_row_dot", "blk_cnt", blk_cnt, ES_I32)), static_cast<float*>(es_op_data("vsa_row_dot", "out", out, ES_F32)), static_cast<int>(es_op_int("vsa_row_dot", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_row_dot", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_row_dot", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_row_dot(const c10::optional<at::Tensor>& x, const c10::optional<at::Tensor>& y, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_tier_b_lists(const c10::optional<at::Tensor>& ab_ptr, const c10::optional<at::Tensor>& ab_idx, const c10::optional<at::Tensor>& a_ptr, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& b_ptr, const c10::optional<at::Tensor>& b_idx, int64_t BH, int64_t NB) {
  const Call es_op_call("vsa_tier_b_lists", {&ab_ptr, &ab_idx, &a_ptr, &bits_a, &b_ptr, &b_idx});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_tier_b_lists", vsa_tier_b_lists(static_cast<const int*>(es_op_data("vsa_tier_b_lists", "ab_ptr", ab_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_tier_b_lists", "ab_idx", ab_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_tier_b_lists", "a_ptr", a_ptr, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_tier_b_lists", "bits_a", bits_a, ES_I32)), static_cast<int*>(es_op_data("vsa_tier_b_lists", "b_ptr", b_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_tier_b_lists", "b_idx", b_idx, ES_I32)), static_cast<int>(es_op_int("vsa_tier_b_lists", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_tier_b_lists", "NB", NB, ES_INT)), es_op_stream));
}
static void meta_vsa_tier_b_lists(const c10::optional<at::Tensor>& ab_ptr, const c10::optional<at::Tensor>& ab_idx, const c10::optional<at::Tensor>& a_ptr, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& b_ptr, const c10::optional<at::Tensor>& b_idx, int64_t BH, int64_t NB) {}

static void op_vsa_pool_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& vr, const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, const c10::optional<at::Tensor>& vc, int64_t BH, int64_t L, int64_t D, int64_t R) {
  const Call es_op_call("vsa_pool_f16", {&q, &k, &v, &blk_cnt, &qr, &kr, &vr, &qc, &kc, &vc});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_pool_f16", vsa_pool_f16(static_cast<const void*>(es_op_data("vsa_pool_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_pool_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_pool_f16", "v", v, ES_HALF)), static_cast<const int*>(es_op_data("vsa_pool_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_pool_f16", "qr", qr, ES_OUT)), static_cast<void*>(es_op_data("vsa_pool_f16", "kr", kr, ES_OUT)), static_cast<void*>(es_op_data("vsa_pool_f16", "vr", vr, ES_OUT)), static_cast<void*>(es_op_data("vsa_pool_f16", "qc", qc, ES_OUT)), static_cast<void*>(es_op_data("vsa_pool_f16", "kc", kc, ES_OUT)), static_cast<void*>(es_op_data("vsa_pool_f16", "vc", vc, ES_OUT)), static_cast<int>(es_op_int("vsa_pool_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_pool_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_pool_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_pool_f16", "R", R, ES_INT)), es_op_stream));
}
static void meta_vsa_pool_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& vr, const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, const c10::optional<at::Tensor>& vc, int64_t BH, int64_t L, int64_t D, int64_t R) {}

static void op_vsa_fuse_fwd_f16(const c10::optional<at::Tensor>& of, const c10::optional<at::Tensor>& oc, const c10::optional<at::Tensor>& gate, const c10::optional<at::Tensor>& o, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D, int64_t NBc_pad, int64_t gate_mode, int64_t gate_act) {
  const Call es_op_call("vsa_fuse_fwd_f16", {&of, &oc, &gate, &o, &blk_cnt});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_fuse_fwd_f16", vsa_fuse_fwd_f16(static_cast<const void*>(es_op_data("vsa_fuse_fwd_f16", "of", of, ES_HALF)), static_cast<const void*>(es_op_data("vsa_fuse_fwd_f16", "oc", oc, ES_HALF)), static_cast<const void*>(es_op_data("vsa_fuse_fwd_f16", "gate", gate, ES_HALF)), static_cast<void*>(es_op_data("vsa_fuse_fwd_f16", "o", o, ES_OUT)), static_cast<const int*>(es_op_data("vsa_fuse_fwd_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<int>(es_op_int("vsa_fuse_fwd_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_fwd_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_fwd_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_fwd_f16", "NBc_pad", NBc_pad, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_fwd_f16", "gate_mode", gate_mode, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_fwd_f16", "gate_act", gate_act, ES_INT)), es_op_stream));
}
static void meta_vsa_fuse_fwd_f16(const c10::optional<at::Tensor>& of, const c10::optional<at::Tensor>& oc, const c10::optional<at::Tensor>& gate, const c10::optional<at::Tensor>& o, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D, int64_t NBc_pad, int64_t gate_mode, int64_t gate_act) {}

static void op_vsa_fuse_bwd_f16(const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& of, const c10::optional<at::Tensor>& oc, const c10::optional<at::Tensor>& gate, const c10::optional<at::Tensor>& dout_f, const c10::optional<at::Tensor>& delta_f, const c10::optional<at::Tensor>& dout_c, const c10::optional<at::Tensor>& delta_c, const c10::optional<at::Tensor>& dgate, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D, int64_t NBc_pad, int64_t gate_mode, int64_t gate_act) {
  const Call es_op_call("vsa_fuse_bwd_f16", {&dout, &of, &oc, &gate, &dout_f, &delta_f, &dout_c, &delta_c, &dgate, &blk_cnt});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_fuse_bwd_f16", vsa_fuse_bwd_f16(static_cast<const void*>(es_op_data("vsa_fuse_bwd_f16", "dout", dout, ES_HALF)), static_cast<const void*>(es_op_data("vsa_fuse_bwd_f16", "of", of, ES_HALF)), static_cast<const void*>(es_op_data("vsa_fuse_bwd_f16", "oc", oc, ES_HALF)), static_cast<const void*>(es_op_data("vsa_fuse_bwd_f16", "gate", gate, ES_HALF)), static_cast<void*>(es_op_data("vsa_fuse_bwd_f16", "dout_f", dout_f, ES_OUT)), static_cast<float*>(es_op_data("vsa_fuse_bwd_f16", "delta_f", delta_f, ES_F32)), static_cast<void*>(es_op_data("vsa_fuse_bwd_f16", "dout_c", dout_c, ES_OUT)), static_cast<float*>(es_op_data("vsa_fuse_bwd_f16", "delta_c", delta_c, ES_F32)), static_cast<void*>(es_op_data("vsa_fuse_bwd_f16", "dgate", dgate, ES_OUT)), static_cast<const int*>(es_op_data("vsa_fuse_bwd_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<int>(es_op_int("vsa_fuse_bwd_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_bwd_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_bwd_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_bwd_f16", "NBc_pad", NBc_pad, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_bwd_f16", "gate_mode", gate_mode, ES_INT)), static_cast<int>(es_op_int("vsa_fuse_bwd_f16", "gate_act", gate_act, ES_INT)), es_op_stream));
}
static void meta_vsa_fuse_bwd_f16(const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& of, const c10::optional<at::Tensor>& oc, const c10::optional<at::Tensor>& gate, const c10::optional<at::Tensor>& dout_f, const c10::optional<at::Tensor>& delta_f, const c10::optional<at::Tensor>& dout_c, const c10::optional<at::Tensor>& delta_c, const c10::optional<at::Tensor>& dgate, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D, int64_t NBc_pad, int64_t gate_mode, int64_t gate_act) {}

static void op_vsa_finalize_f16(const c10::optional<at::Tensor>& acc, const c10::optional<at::Tensor>& add, int64_t add_nb, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_finalize_f16", {&acc, &add, &out, &blk_cnt});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_finalize_f16", vsa_finalize_f16(static_cast<const float*>(es_op_data("vsa_finalize_f16", "acc", acc, ES_F32)), static_cast<const float*>(es_op_data("vsa_finalize_f16", "add", add, ES_F32)), static_cast<int>(es_op_int("vsa_finalize_f16", "add_nb", add_nb, ES_INT)), static_cast<void*>(es_op_data("vsa_finalize_f16", "out", out, ES_OUT)), static_cast<const int*>(es_op_data("vsa_finalize_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<int>(es_op_int("vsa_finalize_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_finalize_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_finalize_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_finalize_f16(const c10::optional<at::Tensor>& acc, const c10::optional<at::Tensor>& add, int64_t add_nb, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& blk_cnt, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_fwd_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& row_ptr, const c10::optional<at::Tensor>& col_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_fwd_f16", {&q, &k, &v, &row_ptr, &col_idx, &blk_cnt, &out, &lse});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_fwd_f16", vsa_attn_fwd_f16(static_cast<const void*>(es_op_data("vsa_attn_fwd_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_fwd_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_fwd_f16", "v", v, ES_HALF)), static_cast<const int*>(es_op_data("vsa_attn_fwd_f16", "row_ptr", row_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_fwd_f16", "col_idx", col_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_fwd_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_attn_fwd_f16", "out", out, ES_OUT)), static_cast<float*>(es_op_data("vsa_attn_fwd_f16", "lse", lse, ES_F32)), static_cast<int>(es_op_int("vsa_attn_fwd_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_fwd_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_fwd_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_fwd_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& row_ptr, const c10::optional<at::Tensor>& col_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_fwd_tasks_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& col_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& part_o, const c10::optional<at::Tensor>& part_lse, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_fwd_tasks_f16", {&q, &k, &v, &col_idx, &blk_cnt, &tasks, &info, &out, &lse, &part_o, &part_lse});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_fwd_tasks_f16", vsa_attn_fwd_tasks_f16(static_cast<const void*>(es_op_data("vsa_attn_fwd_tasks_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_fwd_tasks_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_fwd_tasks_f16", "v", v, ES_HALF)), static_cast<const int*>(es_op_data("vsa_attn_fwd_tasks_f16", "col_idx", col_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_fwd_tasks_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_fwd_tasks_f16", "tasks", tasks, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_fwd_tasks_f16", "info", info, ES_I32)), static_cast<int>(es_op_int("vsa_attn_fwd_tasks_f16", "max_tasks", max_tasks, ES_INT)), static_cast<void*>(es_op_data("vsa_attn_fwd_tasks_f16", "out", out, ES_OUT)), static_cast<float*>(es_op_data("vsa_attn_fwd_tasks_f16", "lse", lse, ES_F32)), static_cast<float*>(es_op_data("vsa_attn_fwd_tasks_f16", "part_o", part_o, ES_F32)), static_cast<float*>(es_op_data("vsa_attn_fwd_tasks_f16", "part_lse", part_lse, ES_F32)), static_cast<int>(es_op_int("vsa_attn_fwd_tasks_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_fwd_tasks_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_fwd_tasks_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_fwd_tasks_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& col_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& part_o, const c10::optional<at::Tensor>& part_lse, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_bwd_kv_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dk, const c10::optional<at::Tensor>& add_dv, int64_t add_nb, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, int64_t out_fp32, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_bwd_kv_f16", {&q, &k, &v, &dout, &lse, &delta, &k2q_ptr, &k2q_idx, &blk_cnt, &add_dk, &add_dv, &dk, &dv});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_bwd_kv_f16", vsa_attn_bwd_kv_f16(static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_f16", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_f16", "dout", dout, ES_HALF)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_f16", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_f16", "delta", delta, ES_F32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_f16", "k2q_ptr", k2q_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_f16", "k2q_idx", k2q_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_f16", "add_dk", add_dk, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_f16", "add_dv", add_dv, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_f16", "add_nb", add_nb, ES_INT)), static_cast<void*>(es_op_data("vsa_attn_bwd_kv_f16", "dk", dk, ES_OUT)), static_cast<void*>(es_op_data("vsa_attn_bwd_kv_f16", "dv", dv, ES_OUT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_f16", "out_fp32", out_fp32, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_bwd_kv_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dk, const c10::optional<at::Tensor>& add_dv, int64_t add_nb, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, int64_t out_fp32, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_bwd_kv_tasks_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& add_dk, const c10::optional<at::Tensor>& add_dv, int64_t add_nb, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, const c10::optional<at::Tensor>& part_dk, const c10::optional<at::Tensor>& part_dv, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_bwd_kv_tasks_f16", {&q, &k, &v, &dout, &lse, &delta, &k2q_idx, &blk_cnt, &tasks, &info, &add_dk, &add_dv, &dk, &dv, &part_dk, &part_dv});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_bwd_kv_tasks_f16", vsa_attn_bwd_kv_tasks_f16(static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "dout", dout, ES_HALF)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "delta", delta, ES_F32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "k2q_idx", k2q_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "tasks", tasks, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "info", info, ES_I32)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_tasks_f16", "max_tasks", max_tasks, ES_INT)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "add_dk", add_dk, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "add_dv", add_dv, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_tasks_f16", "add_nb", add_nb, ES_INT)), static_cast<void*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "dk", dk, ES_OUT)), static_cast<void*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "dv", dv, ES_OUT)), static_cast<float*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "part_dk", part_dk, ES_F32)), static_cast<float*>(es_op_data("vsa_attn_bwd_kv_tasks_f16", "part_dv", part_dv, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_tasks_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_tasks_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_kv_tasks_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_bwd_kv_tasks_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& add_dk, const c10::optional<at::Tensor>& add_dv, int64_t add_nb, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, const c10::optional<at::Tensor>& part_dk, const c10::optional<at::Tensor>& part_dv, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_bwd_q_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq, const c10::optional<at::Tensor>& dq_acc, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_bwd_q_f16", {&q, &k, &v, &dout, &lse, &delta, &q2k_ptr, &q2k_idx, &blk_cnt, &add_dq, &dq, &dq_acc});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_bwd_q_f16", vsa_attn_bwd_q_f16(static_cast<const void*>(es_op_data("vsa_attn_bwd_q_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q_f16", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q_f16", "dout", dout, ES_HALF)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q_f16", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q_f16", "delta", delta, ES_F32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_f16", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_f16", "q2k_idx", q2k_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q_f16", "add_dq", add_dq, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_q_f16", "add_nb", add_nb, ES_INT)), static_cast<void*>(es_op_data("vsa_attn_bwd_q_f16", "dq", dq, ES_OUT)), static_cast<float*>(es_op_data("vsa_attn_bwd_q_f16", "dq_acc", dq_acc, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_q_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_q_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_q_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_bwd_q_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq, const c10::optional<at::Tensor>& dq_acc, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_attn_bwd_q_tasks_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq, const c10::optional<at::Tensor>& part_dq, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_attn_bwd_q_tasks_f16", {&q, &k, &v, &dout, &lse, &delta, &q2k_idx, &blk_cnt, &tasks, &info, &add_dq, &dq, &part_dq});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_attn_bwd_q_tasks_f16", vsa_attn_bwd_q_tasks_f16(static_cast<const void*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "dout", dout, ES_HALF)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "delta", delta, ES_F32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "q2k_idx", q2k_idx, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "tasks", tasks, ES_I32)), static_cast<const int*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "info", info, ES_I32)), static_cast<int>(es_op_int("vsa_attn_bwd_q_tasks_f16", "max_tasks", max_tasks, ES_INT)), static_cast<const float*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "add_dq", add_dq, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_q_tasks_f16", "add_nb", add_nb, ES_INT)), static_cast<void*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "dq", dq, ES_OUT)), static_cast<float*>(es_op_data("vsa_attn_bwd_q_tasks_f16", "part_dq", part_dq, ES_F32)), static_cast<int>(es_op_int("vsa_attn_bwd_q_tasks_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_q_tasks_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_attn_bwd_q_tasks_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_attn_bwd_q_tasks_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& tasks, const c10::optional<at::Tensor>& info, int64_t max_tasks, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq, const c10::optional<at::Tensor>& part_dq, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_block_scores_f16(const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, const c10::optional<at::Tensor>& scores, int64_t NB, int64_t NBc_pad, int64_t bh0, int64_t bh_count, int64_t D) {
  const Call es_op_call("vsa_block_scores_f16", {&qc, &kc, &scores});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_block_scores_f16", vsa_block_scores_f16(static_cast<const void*>(es_op_data("vsa_block_scores_f16", "qc", qc, ES_HALF)), static_cast<const void*>(es_op_data("vsa_block_scores_f16", "kc", kc, ES_HALF)), static_cast<void*>(es_op_data("vsa_block_scores_f16", "scores", scores, ES_OUT)), static_cast<int>(es_op_int("vsa_block_scores_f16", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_block_scores_f16", "NBc_pad", NBc_pad, ES_INT)), static_cast<int>(es_op_int("vsa_block_scores_f16", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_block_scores_f16", "bh_count", bh_count, ES_INT)), static_cast<int>(es_op_int("vsa_block_scores_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_block_scores_f16(const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, const c10::optional<at::Tensor>& scores, int64_t NB, int64_t NBc_pad, int64_t bh0, int64_t bh_count, int64_t D) {}

static void op_vsa_route_rows_f16(const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, int64_t NB, int64_t NBc_pad, int64_t bh0, int64_t bh_count, int64_t K, int64_t D, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {
  const Call es_op_call("vsa_route_rows_f16", {&qc, &kc, &q2k_ptr, &q2k_idx, &k2q_ptr, &k2q_idx, &workspace});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_route_rows_f16", vsa_route_rows_f16(static_cast<const void*>(es_op_data("vsa_route_rows_f16", "qc", qc, ES_HALF)), static_cast<const void*>(es_op_data("vsa_route_rows_f16", "kc", kc, ES_HALF)), static_cast<int>(es_op_int("vsa_route_rows_f16", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_route_rows_f16", "NBc_pad", NBc_pad, ES_INT)), static_cast<int>(es_op_int("vsa_route_rows_f16", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_route_rows_f16", "bh_count", bh_count, ES_INT)), static_cast<int>(es_op_int("vsa_route_rows_f16", "K", K, ES_INT)), static_cast<int>(es_op_int("vsa_route_rows_f16", "D", D, ES_INT)), static_cast<int*>(es_op_data("vsa_route_rows_f16", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_route_rows_f16", "q2k_idx", q2k_idx, ES_I32)), static_cast<int*>(es_op_data("vsa_route_rows_f16", "k2q_ptr", k2q_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_route_rows_f16", "k2q_idx", k2q_idx, ES_I32)), static_cast<void*>(es_op_data("vsa_route_rows_f16", "workspace", workspace, ES_ANY)), static_cast<size_t>(es_op_int("vsa_route_rows_f16", "workspace_bytes", workspace_bytes, ES_SIZE)), es_op_stream));
}
static void meta_vsa_route_rows_f16(const c10::optional<at::Tensor>& qc, const c10::optional<at::Tensor>& kc, int64_t NB, int64_t NBc_pad, int64_t bh0, int64_t bh_count, int64_t K, int64_t D, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {}

static void op_vsa_row_topk_f16(const c10::optional<at::Tensor>& scores, int64_t NB, int64_t bh0, int64_t bh_count, int64_t K, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {
  const Call es_op_call("vsa_row_topk_f16", {&scores, &q2k_ptr, &q2k_idx, &k2q_ptr, &k2q_idx, &workspace});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_row_topk_f16", vsa_row_topk_f16(static_cast<const void*>(es_op_data("vsa_row_topk_f16", "scores", scores, ES_HALF)), static_cast<int>(es_op_int("vsa_row_topk_f16", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_row_topk_f16", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_row_topk_f16", "bh_count", bh_count, ES_INT)), static_cast<int>(es_op_int("vsa_row_topk_f16", "K", K, ES_INT)), static_cast<int*>(es_op_data("vsa_row_topk_f16", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_row_topk_f16", "q2k_idx", q2k_idx, ES_I32)), static_cast<int*>(es_op_data("vsa_row_topk_f16", "k2q_ptr", k2q_ptr, ES_I32)), static_cast<int*>(es_op_data("vsa_row_topk_f16", "k2q_idx", k2q_idx, ES_I32)), static_cast<void*>(es_op_data("vsa_row_topk_f16", "workspace", workspace, ES_ANY)), static_cast<size_t>(es_op_int("vsa_row_topk_f16", "workspace_bytes", workspace_bytes, ES_SIZE)), es_op_stream));
}
static void meta_vsa_row_topk_f16(const c10::optional<at::Tensor>& scores, int64_t NB, int64_t bh0, int64_t bh_count, int64_t K, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& k2q_ptr, const c10::optional<at::Tensor>& k2q_idx, const c10::optional<at::Tensor>& workspace, int64_t workspace_bytes) {}

static void op_vsa_router_lse_f16(const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& lse2, int64_t NB, int64_t R, int64_t BH, int64_t D) {
  const Call es_op_call("vsa_router_lse_f16", {&qr, &kr, &blk_cnt, &lse2});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_router_lse_f16", vsa_router_lse_f16(static_cast<const void*>(es_op_data("vsa_router_lse_f16", "qr", qr, ES_HALF)), static_cast<const void*>(es_op_data("vsa_router_lse_f16", "kr", kr, ES_HALF)), static_cast<const int*>(es_op_data("vsa_router_lse_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<float*>(es_op_data("vsa_router_lse_f16", "lse2", lse2, ES_F32)), static_cast<int>(es_op_int("vsa_router_lse_f16", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_router_lse_f16", "R", R, ES_INT)), static_cast<int>(es_op_int("vsa_router_lse_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_router_lse_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_router_lse_f16(const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& lse2, int64_t NB, int64_t R, int64_t BH, int64_t D) {}

static void op_vsa_router_scores_f16(const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& lse2, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& scores, int64_t NB, int64_t R, int64_t row_norm, int64_t bh0, int64_t bh_count, int64_t D) {
  const Call es_op_call("vsa_router_scores_f16", {&qr, &kr, &lse2, &blk_cnt, &scores});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_router_scores_f16", vsa_router_scores_f16(static_cast<const void*>(es_op_data("vsa_router_scores_f16", "qr", qr, ES_HALF)), static_cast<const void*>(es_op_data("vsa_router_scores_f16", "kr", kr, ES_HALF)), static_cast<const float*>(es_op_data("vsa_router_scores_f16", "lse2", lse2, ES_F32)), static_cast<const int*>(es_op_data("vsa_router_scores_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<float*>(es_op_data("vsa_router_scores_f16", "scores", scores, ES_F32)), static_cast<int>(es_op_int("vsa_router_scores_f16", "NB", NB, ES_INT)), static_cast<int>(es_op_int("vsa_router_scores_f16", "R", R, ES_INT)), static_cast<int>(es_op_int("vsa_router_scores_f16", "row_norm", row_norm, ES_INT)), static_cast<int>(es_op_int("vsa_router_scores_f16", "bh0", bh0, ES_INT)), static_cast<int>(es_op_int("vsa_router_scores_f16", "bh_count", bh_count, ES_INT)), static_cast<int>(es_op_int("vsa_router_scores_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_router_scores_f16(const c10::optional<at::Tensor>& qr, const c10::optional<at::Tensor>& kr, const c10::optional<at::Tensor>& lse2, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& scores, int64_t NB, int64_t R, int64_t row_norm, int64_t bh0, int64_t bh_count, int64_t D) {}

static void op_vsa_split_merge_fwd_f16(const c10::optional<at::Tensor>& part_o, const c10::optional<at::Tensor>& part_lse, const c10::optional<at::Tensor>& merges, const c10::optional<at::Tensor>& info, int64_t max_merges, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& o, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D, int64_t mask_rows) {
  const Call es_op_call("vsa_split_merge_fwd_f16", {&part_o, &part_lse, &merges, &info, &blk_cnt, &o, &lse});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_split_merge_fwd_f16", vsa_split_merge_fwd_f16(static_cast<const float*>(es_op_data("vsa_split_merge_fwd_f16", "part_o", part_o, ES_F32)), static_cast<const float*>(es_op_data("vsa_split_merge_fwd_f16", "part_lse", part_lse, ES_F32)), static_cast<const int*>(es_op_data("vsa_split_merge_fwd_f16", "merges", merges, ES_I32)), static_cast<const int*>(es_op_data("vsa_split_merge_fwd_f16", "info", info, ES_I32)), static_cast<int>(es_op_int("vsa_split_merge_fwd_f16", "max_merges", max_merges, ES_INT)), static_cast<const int*>(es_op_data("vsa_split_merge_fwd_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_split_merge_fwd_f16", "o", o, ES_OUT)), static_cast<float*>(es_op_data("vsa_split_merge_fwd_f16", "lse", lse, ES_F32)), static_cast<int>(es_op_int("vsa_split_merge_fwd_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_split_merge_fwd_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_split_merge_fwd_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_split_merge_fwd_f16", "mask_rows", mask_rows, ES_INT)), es_op_stream));
}
static void meta_vsa_split_merge_fwd_f16(const c10::optional<at::Tensor>& part_o, const c10::optional<at::Tensor>& part_lse, const c10::optional<at::Tensor>& merges, const c10::optional<at::Tensor>& info, int64_t max_merges, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& o, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D, int64_t mask_rows) {}

static void op_vsa_split_merge_sum_f16(const c10::optional<at::Tensor>& part, const c10::optional<at::Tensor>& merges, const c10::optional<at::Tensor>& info, int64_t max_merges, const c10::optional<at::Tensor>& add, int64_t add_nb, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& out_f32, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_split_merge_sum_f16", {&part, &merges, &info, &add, &blk_cnt, &out, &out_f32});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_split_merge_sum_f16", vsa_split_merge_sum_f16(static_cast<const float*>(es_op_data("vsa_split_merge_sum_f16", "part", part, ES_F32)), static_cast<const int*>(es_op_data("vsa_split_merge_sum_f16", "merges", merges, ES_I32)), static_cast<const int*>(es_op_data("vsa_split_merge_sum_f16", "info", info, ES_I32)), static_cast<int>(es_op_int("vsa_split_merge_sum_f16", "max_merges", max_merges, ES_INT)), static_cast<const float*>(es_op_data("vsa_split_merge_sum_f16", "add", add, ES_F32)), static_cast<int>(es_op_int("vsa_split_merge_sum_f16", "add_nb", add_nb, ES_INT)), static_cast<const int*>(es_op_data("vsa_split_merge_sum_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_split_merge_sum_f16", "out", out, ES_OUT)), static_cast<float*>(es_op_data("vsa_split_merge_sum_f16", "out_f32", out_f32, ES_F32)), static_cast<int>(es_op_int("vsa_split_merge_sum_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_split_merge_sum_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_split_merge_sum_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_split_merge_sum_f16(const c10::optional<at::Tensor>& part, const c10::optional<at::Tensor>& merges, const c10::optional<at::Tensor>& info, int64_t max_merges, const c10::optional<at::Tensor>& add, int64_t add_nb, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& out_f32, int64_t BH, int64_t L, int64_t D) {}

static void op_vsa_rep_build_f16(const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, int64_t BH, int64_t L, int64_t D, int64_t RM) {
  const Call es_op_call("vsa_rep_build_f16", {&k, &v, &blk_cnt, &k_mid, &v_mid, &lc_mid, &k_tail, &v_tail, &lc_tail});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_build_f16", vsa_rep_build_f16(static_cast<const void*>(es_op_data("vsa_rep_build_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_build_f16", "v", v, ES_HALF)), static_cast<const int*>(es_op_data("vsa_rep_build_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_rep_build_f16", "k_mid", k_mid, ES_OUT)), static_cast<void*>(es_op_data("vsa_rep_build_f16", "v_mid", v_mid, ES_OUT)), static_cast<float*>(es_op_data("vsa_rep_build_f16", "lc_mid", lc_mid, ES_F32)), static_cast<void*>(es_op_data("vsa_rep_build_f16", "k_tail", k_tail, ES_OUT)), static_cast<void*>(es_op_data("vsa_rep_build_f16", "v_tail", v_tail, ES_OUT)), static_cast<float*>(es_op_data("vsa_rep_build_f16", "lc_tail", lc_tail, ES_F32)), static_cast<int>(es_op_int("vsa_rep_build_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_f16", "RM", RM, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_build_f16(const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, int64_t BH, int64_t L, int64_t D, int64_t RM) {}

static void op_vsa_rep_attn_fwd_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t phases) {
  const Call es_op_call("vsa_rep_attn_fwd_f16", {&q, &k, &v, &k_mid, &v_mid, &lc_mid, &k_tail, &v_tail, &lc_tail, &q2k_ptr, &q2k_idx, &bits_a, &bits_ab, &blk_cnt, &out, &lse});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_attn_fwd_f16", vsa_rep_attn_fwd_f16(static_cast<const void*>(es_op_data("vsa_rep_attn_fwd_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd_f16", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd_f16", "k_mid", k_mid, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd_f16", "v_mid", v_mid, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_attn_fwd_f16", "lc_mid", lc_mid, ES_F32)), static_cast<int>(es_op_int("vsa_rep_attn_fwd_f16", "lc_mid_stride", lc_mid_stride, ES_INT)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd_f16", "k_tail", k_tail, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_fwd_f16", "v_tail", v_tail, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_attn_fwd_f16", "lc_tail", lc_tail, ES_F32)), static_cast<const int*>(es_op_data("vsa_rep_attn_fwd_f16", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_rep_attn_fwd_f16", "q2k_idx", q2k_idx, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_attn_fwd_f16", "bits_a", bits_a, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_attn_fwd_f16", "bits_ab", bits_ab, ES_I32)), static_cast<const int*>(es_op_data("vsa_rep_attn_fwd_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_rep_attn_fwd_f16", "out", out, ES_OUT)), static_cast<float*>(es_op_data("vsa_rep_attn_fwd_f16", "lse", lse, ES_F32)), static_cast<int>(es_op_int("vsa_rep_attn_fwd_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_fwd_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_fwd_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_fwd_f16", "RM", RM, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_fwd_f16", "phases", phases, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_attn_fwd_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, const c10::optional<at::Tensor>& lse, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t phases) {}

static void op_vsa_rep_attn_bwd_q_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq_acc, const c10::optional<at::Tensor>& dq, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t phases) {
  const Call es_op_call("vsa_rep_attn_bwd_q_f16", {&q, &k, &v, &k_mid, &v_mid, &lc_mid, &k_tail, &v_tail, &lc_tail, &dout, &lse, &delta, &q2k_ptr, &q2k_idx, &bits_a, &bits_ab, &blk_cnt, &add_dq, &dq_acc, &dq});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_attn_bwd_q_f16", vsa_rep_attn_bwd_q_f16(static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q_f16", "v", v, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q_f16", "k_mid", k_mid, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q_f16", "v_mid", v_mid, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q_f16", "lc_mid", lc_mid, ES_F32)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q_f16", "lc_mid_stride", lc_mid_stride, ES_INT)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q_f16", "k_tail", k_tail, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q_f16", "v_tail", v_tail, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q_f16", "lc_tail", lc_tail, ES_F32)), static_cast<const void*>(es_op_data("vsa_rep_attn_bwd_q_f16", "dout", dout, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q_f16", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q_f16", "delta", delta, ES_F32)), static_cast<const int*>(es_op_data("vsa_rep_attn_bwd_q_f16", "q2k_ptr", q2k_ptr, ES_I32)), static_cast<const int*>(es_op_data("vsa_rep_attn_bwd_q_f16", "q2k_idx", q2k_idx, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_attn_bwd_q_f16", "bits_a", bits_a, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_attn_bwd_q_f16", "bits_ab", bits_ab, ES_I32)), static_cast<const int*>(es_op_data("vsa_rep_attn_bwd_q_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q_f16", "add_dq", add_dq, ES_F32)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q_f16", "add_nb", add_nb, ES_INT)), static_cast<const float*>(es_op_data("vsa_rep_attn_bwd_q_f16", "dq_acc", dq_acc, ES_F32)), static_cast<void*>(es_op_data("vsa_rep_attn_bwd_q_f16", "dq", dq, ES_OUT)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q_f16", "RM", RM, ES_INT)), static_cast<int>(es_op_int("vsa_rep_attn_bwd_q_f16", "phases", phases, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_attn_bwd_q_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& q2k_ptr, const c10::optional<at::Tensor>& q2k_idx, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& add_dq, int64_t add_nb, const c10::optional<at::Tensor>& dq_acc, const c10::optional<at::Tensor>& dq, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t phases) {}

static void op_vsa_rep_bwd_tables_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& k_tab, const c10::optional<at::Tensor>& v_tab, const c10::optional<at::Tensor>& lc, int64_t lc_stride, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& dk_tab, const c10::optional<at::Tensor>& dv_tab, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t tier) {
  const Call es_op_call("vsa_rep_bwd_tables_f16", {&q, &dout, &k_tab, &v_tab, &lc, &lse, &delta, &bits_a, &bits_ab, &dk_tab, &dv_tab});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_bwd_tables_f16", vsa_rep_bwd_tables_f16(static_cast<const void*>(es_op_data("vsa_rep_bwd_tables_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_tables_f16", "dout", dout, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_tables_f16", "k_tab", k_tab, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_tables_f16", "v_tab", v_tab, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_bwd_tables_f16", "lc", lc, ES_F32)), static_cast<int>(es_op_int("vsa_rep_bwd_tables_f16", "lc_stride", lc_stride, ES_INT)), static_cast<const float*>(es_op_data("vsa_rep_bwd_tables_f16", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_bwd_tables_f16", "delta", delta, ES_F32)), static_cast<const unsigned*>(es_op_data("vsa_rep_bwd_tables_f16", "bits_a", bits_a, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_bwd_tables_f16", "bits_ab", bits_ab, ES_I32)), static_cast<float*>(es_op_data("vsa_rep_bwd_tables_f16", "dk_tab", dk_tab, ES_F32)), static_cast<float*>(es_op_data("vsa_rep_bwd_tables_f16", "dv_tab", dv_tab, ES_F32)), static_cast<int>(es_op_int("vsa_rep_bwd_tables_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_tables_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_tables_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_tables_f16", "RM", RM, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_tables_f16", "tier", tier, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_bwd_tables_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& k_tab, const c10::optional<at::Tensor>& v_tab, const c10::optional<at::Tensor>& lc, int64_t lc_stride, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& dk_tab, const c10::optional<at::Tensor>& dv_tab, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t tier) {}

static void op_vsa_rep_bwd_both_tables_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& dk_mid, const c10::optional<at::Tensor>& dv_mid, const c10::optional<at::Tensor>& dk_tail, const c10::optional<at::Tensor>& dv_tail, int64_t BH, int64_t L, int64_t D, int64_t RM) {
  const Call es_op_call("vsa_rep_bwd_both_tables_f16", {&q, &dout, &k_mid, &v_mid, &lc_mid, &k_tail, &v_tail, &lc_tail, &lse, &delta, &bits_a, &bits_ab, &dk_mid, &dv_mid, &dk_tail, &dv_tail});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_bwd_both_tables_f16", vsa_rep_bwd_both_tables_f16(static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables_f16", "q", q, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables_f16", "dout", dout, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables_f16", "k_mid", k_mid, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables_f16", "v_mid", v_mid, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_bwd_both_tables_f16", "lc_mid", lc_mid, ES_F32)), static_cast<int>(es_op_int("vsa_rep_bwd_both_tables_f16", "lc_mid_stride", lc_mid_stride, ES_INT)), static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables_f16", "k_tail", k_tail, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_bwd_both_tables_f16", "v_tail", v_tail, ES_HALF)), static_cast<const float*>(es_op_data("vsa_rep_bwd_both_tables_f16", "lc_tail", lc_tail, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_bwd_both_tables_f16", "lse", lse, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_bwd_both_tables_f16", "delta", delta, ES_F32)), static_cast<const unsigned*>(es_op_data("vsa_rep_bwd_both_tables_f16", "bits_a", bits_a, ES_I32)), static_cast<const unsigned*>(es_op_data("vsa_rep_bwd_both_tables_f16", "bits_ab", bits_ab, ES_I32)), static_cast<float*>(es_op_data("vsa_rep_bwd_both_tables_f16", "dk_mid", dk_mid, ES_F32)), static_cast<float*>(es_op_data("vsa_rep_bwd_both_tables_f16", "dv_mid", dv_mid, ES_F32)), static_cast<float*>(es_op_data("vsa_rep_bwd_both_tables_f16", "dk_tail", dk_tail, ES_F32)), static_cast<float*>(es_op_data("vsa_rep_bwd_both_tables_f16", "dv_tail", dv_tail, ES_F32)), static_cast<int>(es_op_int("vsa_rep_bwd_both_tables_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_both_tables_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_both_tables_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_bwd_both_tables_f16", "RM", RM, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_bwd_both_tables_f16(const c10::optional<at::Tensor>& q, const c10::optional<at::Tensor>& dout, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, int64_t lc_mid_stride, const c10::optional<at::Tensor>& k_tail, const c10::optional<at::Tensor>& v_tail, const c10::optional<at::Tensor>& lc_tail, const c10::optional<at::Tensor>& lse, const c10::optional<at::Tensor>& delta, const c10::optional<at::Tensor>& bits_a, const c10::optional<at::Tensor>& bits_ab, const c10::optional<at::Tensor>& dk_mid, const c10::optional<at::Tensor>& dv_mid, const c10::optional<at::Tensor>& dk_tail, const c10::optional<at::Tensor>& dv_tail, int64_t BH, int64_t L, int64_t D, int64_t RM) {}

static void op_vsa_rep_build_kmeans_f16(const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& labels, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t iters, int64_t seed) {
  const Call es_op_call("vsa_rep_build_kmeans_f16", {&k, &v, &blk_cnt, &k_mid, &v_mid, &lc_mid, &counts, &labels});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_build_kmeans_f16", vsa_rep_build_kmeans_f16(static_cast<const void*>(es_op_data("vsa_rep_build_kmeans_f16", "k", k, ES_HALF)), static_cast<const void*>(es_op_data("vsa_rep_build_kmeans_f16", "v", v, ES_HALF)), static_cast<const int*>(es_op_data("vsa_rep_build_kmeans_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<void*>(es_op_data("vsa_rep_build_kmeans_f16", "k_mid", k_mid, ES_OUT)), static_cast<void*>(es_op_data("vsa_rep_build_kmeans_f16", "v_mid", v_mid, ES_OUT)), static_cast<float*>(es_op_data("vsa_rep_build_kmeans_f16", "lc_mid", lc_mid, ES_F32)), static_cast<int*>(es_op_data("vsa_rep_build_kmeans_f16", "counts", counts, ES_I32)), static_cast<uint8_t*>(es_op_data("vsa_rep_build_kmeans_f16", "labels", labels, ES_U8)), static_cast<int>(es_op_int("vsa_rep_build_kmeans_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_kmeans_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_kmeans_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_kmeans_f16", "RM", RM, ES_INT)), static_cast<int>(es_op_int("vsa_rep_build_kmeans_f16", "iters", iters, ES_INT)), static_cast<unsigned>(es_op_int("vsa_rep_build_kmeans_f16", "seed", seed, ES_UINT)), es_op_stream));
}
static void meta_vsa_rep_build_kmeans_f16(const c10::optional<at::Tensor>& k, const c10::optional<at::Tensor>& v, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& k_mid, const c10::optional<at::Tensor>& v_mid, const c10::optional<at::Tensor>& lc_mid, const c10::optional<at::Tensor>& counts, const c10::optional<at::Tensor>& labels, int64_t BH, int64_t L, int64_t D, int64_t RM, int64_t iters, int64_t seed) {}

static void op_vsa_rep_unpool_f16(const c10::optional<at::Tensor>& acc_k, const c10::optional<at::Tensor>& acc_v, const c10::optional<at::Tensor>& dk_mid, const c10::optional<at::Tensor>& dv_mid, const c10::optional<at::Tensor>& dk_tail, const c10::optional<at::Tensor>& dv_tail, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& labels, const c10::optional<at::Tensor>& mid_counts, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, int64_t BH, int64_t L, int64_t D, int64_t RM) {
  const Call es_op_call("vsa_rep_unpool_f16", {&acc_k, &acc_v, &dk_mid, &dv_mid, &dk_tail, &dv_tail, &blk_cnt, &labels, &mid_counts, &dk, &dv});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_rep_unpool_f16", vsa_rep_unpool_f16(static_cast<const float*>(es_op_data("vsa_rep_unpool_f16", "acc_k", acc_k, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_unpool_f16", "acc_v", acc_v, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_unpool_f16", "dk_mid", dk_mid, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_unpool_f16", "dv_mid", dv_mid, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_unpool_f16", "dk_tail", dk_tail, ES_F32)), static_cast<const float*>(es_op_data("vsa_rep_unpool_f16", "dv_tail", dv_tail, ES_F32)), static_cast<const int*>(es_op_data("vsa_rep_unpool_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<const uint8_t*>(es_op_data("vsa_rep_unpool_f16", "labels", labels, ES_U8)), static_cast<const int*>(es_op_data("vsa_rep_unpool_f16", "mid_counts", mid_counts, ES_I32)), static_cast<void*>(es_op_data("vsa_rep_unpool_f16", "dk", dk, ES_OUT)), static_cast<void*>(es_op_data("vsa_rep_unpool_f16", "dv", dv, ES_OUT)), static_cast<int>(es_op_int("vsa_rep_unpool_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_rep_unpool_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_rep_unpool_f16", "D", D, ES_INT)), static_cast<int>(es_op_int("vsa_rep_unpool_f16", "RM", RM, ES_INT)), es_op_stream));
}
static void meta_vsa_rep_unpool_f16(const c10::optional<at::Tensor>& acc_k, const c10::optional<at::Tensor>& acc_v, const c10::optional<at::Tensor>& dk_mid, const c10::optional<at::Tensor>& dv_mid, const c10::optional<at::Tensor>& dk_tail, const c10::optional<at::Tensor>& dv_tail, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& labels, const c10::optional<at::Tensor>& mid_counts, const c10::optional<at::Tensor>& dk, const c10::optional<at::Tensor>& dv, int64_t BH, int64_t L, int64_t D, int64_t RM) {}

static void op_vsa_row_dot_f16(const c10::optional<at::Tensor>& x, const c10::optional<at::Tensor>& y, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, int64_t BH, int64_t L, int64_t D) {
  const Call es_op_call("vsa_row_dot_f16", {&x, &y, &blk_cnt, &out});
  c10::OptionalDeviceGuard es_op_guard(es_op_call.dev);
  const hipStream_t es_op_stream =
      es_op_call.dev ? c10::hip::getCurrentHIPStream(es_op_call.dev->index()).stream() : nullptr;
  es_op_check("vsa_row_dot_f16", vsa_row_dot_f16(static_cast<const void*>(es_op_data("vsa_row_dot_f16", "x", x, ES_HALF)), static_cast<const void*>(es_op_data("vsa_row_dot_f16", "y", y, ES_HALF)), static_cast<const int*>(es_op_data("vsa_row_dot_f16", "blk_cnt", blk_cnt, ES_I32)), static_cast<float*>(es_op_data("vsa_row_dot_f16", "out", out, ES_F32)), static_cast<int>(es_op_int("vsa_row_dot_f16", "BH", BH, ES_INT)), static_cast<int>(es_op_int("vsa_row_dot_f16", "L", L, ES_INT)), static_cast<int>(es_op_int("vsa_row_dot_f16", "D", D, ES_INT)), es_op_stream));
}
static void meta_vsa_row_dot_f16(const c10::optional<at::Tensor>& x, const c10::optional<at::Tensor>& y, const c10::optional<at::Tensor>& blk_cnt, const c10::optional<at::Tensor>& out, int64_t BH, int64_t L, int64_t D) {}

TORCH_LIBRARY(echosparse_gfx950, m) {
  m.def("es_block_attention(Tensor? q, Tensor? k, Tensor? v, Tensor(a!)? out, Tensor? counts, Tensor? blocks, int nk, Tensor? offset, Tensor(b!)? lse, Tensor(c!)? flags, Tensor(d!)? mass, float threshold, int L, int H, int D) -> ()");
  m.def("es_sparse_attention(Tensor? q, Tensor? k, Tensor? v, Tensor? k_mean, Tensor? v_mean, Tensor? means, Tensor? mean_counts, Tensor(a!)? out, Tensor? counts, Tensor? blocks, int nk, Tensor? offset, Tensor(b!)? lse, Tensor(c!)? flags, Tensor? refine, Tensor? refine_counts, int rw, Tensor? k_rep, Tensor? v_rep, Tensor? log_counts, Tensor(d!)? mass, float threshold, int tiles, int L, int H, int D) -> ()");
  m.def("es_exact_fallback(Tensor? q, Tensor? k, Tensor? v, Tensor(a!)? out, Tensor? counts, Tensor? blocks, int nk, Tensor(b!)? lse, Tensor? flags, int L, int H, int D) -> ()");
  m.def("es_compensate_fallback(Tensor? q, Tensor? k_mean, Tensor? v_mean, Tensor? keep, Tensor(a!)? lse, Tensor(b!)? out, Tensor? flags, int L, int H, int D) -> ()");
  m.def("es_dense_attention(Tensor? q, Tensor? k, Tensor? v, Tensor(a!)? out, Tensor(b!)? lse2, int L, int H, int D) -> ()");
  m.def("es_dense_attention_kv(Tensor? q, Tensor? k, Tensor? v, Tensor(a!)? out, Tensor(b!)? lse2, int Lq, int Lk, int H, int D) -> ()");
  m.def("es_dense_attention_ws(Tensor? q, Tensor? k, Tensor? v, Tensor(a!)? out, Tensor(b!)? lse2, Tensor(c!)? workspace, int workspace_bytes, int Lq, int Lk, int H, int D) -> ()");
  m.def("es_block_means(Tensor? k, Tensor? v, Tensor(a!)? k_mean, Tensor(b!)? v_mean, int L, int H, int D) -> ()");
  m.def("es_estimate_skipped(Tensor? q, Tensor? k_mean, Tensor? keep, Tensor? offset, Tensor? lse, Tensor(a!)? mass, Tensor(b!)? scale_exact, Tensor(c!)? scale_skip, int L, int H, int D) -> ()");
  m.def("es_full_step_scales(Tensor? offset, Tensor(a!)? lse, Tensor(b!)? scale_exact, Tensor(c!)? scale_skip, int L, int H) -> ()");
  m.def("es_select_blocks(Tensor? mass, Tensor? keep_prev, Tensor? scale_exact, Tensor? scale_skip, Tensor(a!)? keep, Tensor(b!)? counts, Tensor(c!)? blocks, Tensor? flags, Tensor(d!)? skip_bits, int nw, Tensor(e!)? refine, int rw, int k, int r, int L, int H, int sink) -> ()");
  m.def("es_pack_plan(Tensor? keep, Tensor(a!)? exact_bits, int nw, int H, int nq, int nb) -> ()");
  m.def("es_rebuild_plan(Tensor? exact_bits, Tensor? skip_bits, int nw, Tensor(a!)? keep, Tensor(b!)? counts, Tensor(c!)? blocks, Tensor(d!)? refine, Tensor(e!)? refine_counts, int rw, Tensor(f!)? means, Tensor(g!)? mean_counts, int H, int nq, int nb) -> ()");
  m.def("es_representatives(Tensor? q, Tensor? k, Tensor? v, Tensor(a!)? k_rep, Tensor(b!)? v_rep, Tensor(c!)? log_counts, Tensor(d!)? k_mean, Tensor(e!)? v_mean, Tensor(f!)? workspace, int workspace_bytes, int iters, int L, int H, int D) -> ()");
  m.def("es_representatives_noalloc(Tensor? q, Tensor? k, Tensor? v, Tensor(a!)? k_rep, Tensor(b!)? v_rep, Tensor(c!)? log_counts, Tensor(d!)? k_mean, Tensor(e!)? v_mean, int iters, int L, int H, int D) -> ()");
  m.def("vsa_pool(Tensor? q, Tensor? k, Tensor? v, Tensor? blk_cnt, Tensor(a!)? qr, Tensor(b!)? kr, Tensor(c!)? vr, Tensor(d!)? qc, Tensor(e!)? kc, Tensor(f!)? vc, int BH, int L, int D, int R) -> ()");
  m.def("vsa_fuse_fwd(Tensor? of, Tensor? oc, Tensor? gate, Tensor(a!)? o, Tensor? blk_cnt, int BH, int L, int D, int NBc_pad, int gate_mode, int gate_act) -> ()");
  m.def("vsa_fuse_bwd(Tensor? dout, Tensor? of, Tensor? oc, Tensor? gate, Tensor(a!)? dout_f, Tensor(b!)? delta_f, Tensor(c!)? dout_c, Tensor(d!)? delta_c, Tensor(e!)? dgate, Tensor? blk_cnt, int BH, int L, int D, int NBc_pad, int gate_mode, int gate_act) -> ()");
  m.def("vsa_finalize(Tensor? acc, Tensor? add, int add_nb, Tensor(a!)? out, Tensor? blk_cnt, int BH, int L, int D) -> ()");
  m.def("vsa_attn_fwd(Tensor? q, Tensor? k, Tensor? v, Tensor? row_ptr, Tensor? col_idx, Tensor? blk_cnt, Tensor(a!)? out, Tensor(b!)? lse, int BH, int L, int D) -> ()");
  m.def("vsa_attn_fwd_tasks(Tensor? q, Tensor? k, Tensor? v, Tensor? col_idx, Tensor? blk_cnt, Tensor? tasks, Tensor? info, int max_tasks, Tensor(a!)? out, Tensor(b!)? lse, Tensor(c!)? part_o, Tensor(d!)? part_lse, int BH, int L, int D) -> ()");
  m.def("vsa_attn_bwd_kv(Tensor? q, Tensor? k, Tensor? v, Tensor? dout, Tensor? lse, Tensor? delta, Tensor? k2q_ptr, Tensor? k2q_idx, Tensor? blk_cnt, Tensor? add_dk, Tensor? add_dv, int add_nb, Tensor(a!)? dk, Tensor(b!)? dv, int out_fp32, int BH, int L, int D) -> ()");
  m.def("vsa_attn_bwd_kv_tasks(Tensor? q, Tensor? k, Tensor? v, Tensor? dout, Tensor? lse, Tensor? delta, Tensor? k2q_idx, Tensor? blk_cnt, Tensor? tasks, Tensor? info, int max_tasks, Tensor? add_dk, Tensor? add_dv, int add_nb, Tensor(a!)? dk, Tensor(b!)? dv, Tensor(c!)? part_dk, Tensor(d!)? part_dv, int BH, int L, int D) -> ()");
  m.def("vsa_attn_bwd_q(Tensor? q, Tensor? k, Tensor? v, Tensor? dout, Tensor? lse, Tensor? delta, Tensor? q2k_ptr, Tensor? q2k_idx, Tensor? blk_cnt, Tensor? add_dq, int add_nb, Tensor(a!)? dq, Tensor(b!)? dq_acc, int BH, int L, int D) -> ()");
  m.def("vsa_attn_bwd_q_tasks(Tensor? q, Tensor? k, Tensor? v, Tensor? dout, Tensor? lse, Tensor? delta, Tensor? q2k_idx, Tensor? blk_cnt, Tensor? tasks, Tensor? info, int max_tasks, Tensor? add_dq, int add_nb, Tensor(a!)? dq, Tensor(b!)? part_dq, int BH, int L, int D) -> ()");
  m.def("vsa_block_scores(Tensor? qc, Tensor? kc, Tensor(a!)? scores, int NB, int NBc_pad, int bh0, int bh_count, int D) -> ()");
  m.def("vsa_route_rows(Tensor? qc, Tensor? kc, int NB, int NBc_pad, int bh0, int bh_count, int K, int D, Tensor(a!)? q2k_ptr, Tensor(b!)? q2k_idx, Tensor(c!)? k2q_ptr, Tensor(d!)? k2q_idx, Tensor(e!)? workspace, int workspace_bytes) -> ()");
  m.def("vsa_row_topk(Tensor? scores, int NB, int bh0, int bh_count, int K, Tensor(a!)? q2k_ptr, Tensor(b!)? q2k_idx, Tensor(c!)? k2q_ptr, Tensor(d!)? k2q_idx, Tensor(e!)? workspace, int workspace_bytes) -> ()");
  m.def("vsa_router_lse(Tensor? qr, Tensor? kr, Tensor? blk_cnt, Tensor(a!)? lse2, int NB, int R, int BH, int D) -> ()");
  m.def("vsa_router_scores(Tensor? qr, Tensor? kr, Tensor? lse2, Tensor? blk_cnt, Tensor(a!)? scores, int NB, int R, int row_norm, int bh0, int bh_count, int D) -> ()");
  m.def("vsa_global_topk(Tensor? scores, int NB, int bh0, int bh_count, int budget, Tensor(a!)? q2k_ptr, Tensor(b!)? q2k_idx, Tensor(c!)? k2q_ptr, Tensor(d!)? k2q_idx, Tensor(e!)? bits_out, Tensor(f!)? workspace, int workspace_bytes) -> ()");
  m.def("vsa_csr_transpose(Tensor? ptr, Tensor? idx, int NB, int bh0, int bh_count, Tensor(a!)? out_ptr, Tensor(b!)? out_idx, Tensor(c!)? workspace, int workspace_bytes) -> ()");
  m.def("vsa_dense_lists(int NB, int BH, Tensor(a!)? cnt, Tensor(b!)? ptr, Tensor(c!)? idx) -> ()");
  m.def("vsa_split_plan(Tensor? ptr, int BH, int NB, int chunk, int max_slots, int min_len, float rel_mean, float tail_frac, int resident, int budget, Tensor(a!)? tasks, Tensor(b!)? merges, Tensor(c!)? info) -> ()");
  m.def("vsa_split_merge_fwd(Tensor? part_o, Tensor? part_lse, Tensor? merges, Tensor? info, int max_merges, Tensor? blk_cnt, Tensor(a!)? o, Tensor(b!)? lse, int BH, int L, int D, int mask_rows) -> ()");
  m.def("vsa_split_merge_sum(Tensor? part, Tensor? merges, Tensor? info, int max_merges, Tensor? add, int add_nb, Tensor? blk_cnt, Tensor(a!)? out, Tensor(b!)? out_f32, int BH, int L, int D) -> ()");
  m.def("vsa_rep_build(Tensor? k, Tensor? v, Tensor? blk_cnt, Tensor(a!)? k_mid, Tensor(b!)? v_mid, Tensor(c!)? lc_mid, Tensor(d!)? k_tail, Tensor(e!)? v_tail, Tensor(f!)? lc_tail, int BH, int L, int D, int RM) -> ()");
  m.def("vsa_rep_build_kmeans(Tensor? k, Tensor? v, Tensor? blk_cnt, Tensor(a!)? k_mid, Tensor(b!)? v_mid, Tensor(c!)? lc_mid, Tensor(d!)? counts, Tensor(e!)? labels, int BH, int L, int D, int RM, int iters, int seed) -> ()");
  m.def("vsa_row_tiers(Tensor? scores, int NB, int bh0, int bh_count, int ka, int kab, Tensor(a!)? a_ptr, Tensor(b!)? a_idx, Tensor(c!)? ab_ptr, Tensor(d!)? ab_idx, Tensor(e!)? bits_a, Tensor(f!)? bits_ab) -> ()");
  m.def("vsa_rep_attn_fwd(Tensor? q, Tensor? k, Tensor? v, Tensor? k_mid, Tensor? v_mid, Tensor? lc_mid, int lc_mid_stride, Tensor? k_tail, Tensor? v_tail, Tensor? lc_tail, Tensor? q2k_ptr, Tensor? q2k_idx, Tensor? bits_a, Tensor? bits_ab, Tensor? blk_cnt, Tensor(a!)? out, Tensor(b!)? lse, int BH, int L, int D, int RM, int phases) -> ()");
  m.def("vsa_rep_attn_bwd_q(Tensor? q, Tensor? k, Tensor? v, Tensor? k_mid, Tensor? v_mid, Tensor? lc_mid, int lc_mid_stride, Tensor? k_tail, Tensor? v_tail, Tensor? lc_tail, Tensor? dout, Tensor? lse, Tensor? delta, Tensor? q2k_ptr, Tensor? q2k_idx, Tensor? bits_a, Tensor? bits_ab, Tensor? blk_cnt, Tensor? add_dq, int add_nb, Tensor? dq_acc, Tensor(a!)? dq, int BH, int L, int D, int RM, int phases) -> ()");
  m.def("vsa_rep_bwd_tables(Tensor? q, Tensor? dout, Tensor? k_tab, Tensor? v_tab, Tensor? lc, int lc_stride, Tensor? lse, Tensor? delta, Tensor? bits_a, Tensor? bits_ab, Tensor(a!)? dk_tab, Tensor(b!)? dv_tab, int BH, int L, int D, int RM, int tier) -> ()");
  m.def("vsa_rep_bwd_both_tables(Tensor? q, Tensor? dout, Tensor? k_mid, Tensor? v_mid, Tensor? lc_mid, int lc_mid_stride, Tensor? k_tail, Tensor? v_tail, Tensor? lc_tail, Tensor? lse, Tensor? delta, Tensor? bits_a, Tensor? bits_ab, Tensor(a!)? dk_mid, Tensor(b!)? dv_mid, Tensor(c!)? dk_tail, Tensor(d!)? dv_tail, int BH, int L, int D, int RM) -> ()");
  m.def("vsa_rep_unpool(Tensor? acc_k, Tensor? acc_v, Tensor? dk_mid, Tensor? dv_mid, Tensor? dk_tail, Tensor? dv_tail, Tensor? blk_cnt, Tensor? labels, Tensor? mid_counts, Tensor(a!)? dk, Tensor(b!)? dv, int BH, int L, int D, int RM) -> ()");
  m.def("vsa_row_dot(Tensor? x, Tensor? y, Tensor? blk_cnt, Tensor(a!)? out, int BH, int L, int D) -> ()");
  m.def("vsa_tier_b_lists(Tensor? ab_ptr, Tensor? ab_idx, Tensor? a_ptr, Tensor? bits_a, Tensor(a!)? b_ptr, Tensor(b!)? b_idx, int BH, int NB) -> ()");
  m.def("vsa_pool_f16(Tensor? q, Tensor? k, Tensor? v, Tensor? blk_cnt, Tensor(a!)? qr, Tensor(b!)? kr, Tensor(c!)? vr, Tensor(d!)? qc, Tensor(e!)? kc, Tensor(f!)? vc, int BH, int L, int D, int R) -> ()");
  m.def("vsa_fuse_fwd_f16(Tensor? of, Tensor? oc, Tensor? gate, Tensor(a!)? o, Tensor? blk_cnt, int BH, int L, int D, int NBc_pad, int gate_mode, int gate_act) -> ()");
  m.def("vsa_fuse_bwd_f16(Tensor? dout, Tensor? of, Tensor? oc, Tensor? gate, Tensor(a!)? dout_f, Tensor(b!)? delta_f, Tensor(c!)? dout_c, Tensor(d!)? delta_c, Tensor(e!)? dgate, Tensor? blk_cnt, int BH, int L, int D, int NBc_pad, int gate_mode, int gate_act) -> ()");
  m.def("vsa_finalize_f16(Tensor? acc, Tensor? add, int add_nb, Tensor(a!)? out, Tensor? blk_cnt, int BH, int L, int D) -> ()");
  m.def("vsa_attn_fwd_f16(Tensor? q, Tensor? k, Tensor? v, Tensor? row_ptr, Tensor? col_idx, Tensor? blk_cnt, Tensor(a!)? out, Tensor(b!)? lse, int BH, int L, int D) -> ()");
  m.def("vsa_attn_fwd_tasks_f16(Tensor? q, Tensor? k, Tensor? v, Tensor? col_idx, Tensor? blk_cnt, Tensor? tasks, Tensor? info, int max_tasks, Tensor(a!)? out, Tensor(b!)? lse, Tensor(c!)? part_o, Tensor(d!)? part_lse, int BH, int L, int D) -> ()");
  m.def("vsa_attn_bwd_kv_f16(Tensor? q, Tensor? k, Tensor? v, Tensor? dout, Tensor? lse, Tensor? delta, Tensor? k2q_ptr, Tensor? k2q_idx, Tensor? blk_cnt, Tensor? add_dk, Tensor? add_dv, int add_nb, Tensor(a!)? dk, Tensor(b!)? dv, int out_fp32, int BH, int L, int D) -> ()");
  m.def("vsa_attn_bwd_kv_tasks_f16(Tensor? q, Tensor? k, Tensor? v, Tensor? dout, Tensor? lse, Tensor? delta, Tensor? k2q_idx, Tensor? blk_cnt, Tensor? tasks, Tensor? info, int max_tasks, Tensor? add_dk, Tensor? add_dv, int add_nb, Tensor(a!)? dk, Tensor(b!)? dv, Tensor(c!)? part_dk, Tensor(d!)? part_dv, int BH, int L, int D) -> ()");
  m.def("vsa_attn_bwd_q_f16(Tensor? q, Tensor? k, Tensor? v, Tensor? dout, Tensor? lse, Tensor? delta, Tensor? q2k_ptr, Tensor? q2k_idx, Tensor? blk_cnt, Tensor? add_dq, int add_nb, Tensor(a!)? dq, Tensor(b!)? dq_acc, int BH, int L, int D) -> ()");
  m.def("vsa_attn_bwd_q_tasks_f16(Tensor? q, Tensor? k, Tensor? v, Tensor? dout, Tensor? lse, Tensor? delta, Tensor? q2k_idx, Tensor? blk_cnt, Tensor? tasks, Tensor? info, int max_tasks, Tensor? add_dq, int add_nb, Tensor(a!)? dq, Tensor(b!)? part_dq, int BH, int L, int D) -> ()");
  m.def("vsa_block_scores_f16(Tensor? qc, Tensor? kc, Tensor(a!)? scores, int NB, int NBc_pad, int bh0, int bh_count, int D) -> ()");
  m.def("vsa_route_rows_f16(Tensor? qc, Tensor? kc, int NB, int NBc_pad, int bh0, int bh_count, int K, int D, Tensor(a!)? q2k_ptr, Tensor(b!)? q2k_idx, Tensor(c!)? k2q_ptr, Tensor(d!)? k2q_idx, Tensor(e!)? workspace, int workspace_bytes) -> ()");
  m.def("vsa_row_topk_f16(Tensor? scores, int NB, int bh0, int bh_count, int K, Tensor(a!)? q2k_ptr, Tensor(b!)? q2k_idx, Tensor(c!)? k2q_ptr, Tensor(d!)? k2q_idx, Tensor(e!)? workspace, int workspace_bytes) -> ()");
  m.def("vsa_router_lse_f16(Tensor? qr, Tensor? kr, Tensor? blk_cnt, Tensor(a!)? lse2, int NB, int R, int BH, int D) -> ()");
  m.def("vsa_router_scores_f16(Tensor? qr, Tensor? kr, Tensor? lse2, Tensor? blk_cnt, Tensor(a!)? scores, int NB, int R, int row_norm, int bh0, int bh_count, int D) -> ()");
  m.def("vsa_split_merge_fwd_f16(Tensor? part_o, Tensor? part_lse, Tensor? merges, Tensor? info, int max_merges, Tensor? blk_cnt, Tensor(a!)? o, Tensor(b!)? lse, int BH, int L, int D, int mask_rows) -> ()");
  m.def("vsa_split_merge_sum_f16(Tensor? part, Tensor? merges, Tensor? info, int max_merges, Tensor? add, int add_nb, Tensor? blk_cnt, Tensor(a!)? out, Tensor(b!)? out_f32, int BH, int L, int D) -> ()");
  m.def("vsa_rep_build_f16(Tensor? k, Tensor? v, Tensor? blk_cnt, Tensor(a!)? k_mid, Tensor(b!)? v_mid, Tensor(c!)? lc_mid, Tensor(d!)? k_tail, Tensor(e!)? v_tail, Tensor(f!)? lc_tail, int BH, int L, int D, int RM) -> ()");
  m.def("vsa_rep_attn_fwd_f16(Tensor? q, Tensor? k, Tensor? v, Tensor? k_mid, Tensor? v_mid, Tensor? lc_mid, int lc_mid_stride, Tensor? k_tail, Tensor? v_tail, Tensor? lc_tail, Tensor? q2k_ptr, Tensor? q2k_idx, Tensor? bits_a, Tensor? bits_ab, Tensor? blk_cnt, Tensor(a!)? out, Tensor(b!)? lse, int BH, int L, int D, int RM, int phases) -> ()");
  m.def("vsa_rep_attn_bwd_q_f16(Tensor? q, Tensor? k, Tensor? v, Tensor? k_mid, Tensor? v_mid, Tensor? lc_mid, int lc_mid_stride, Tensor? k_tail, Tensor? v_tail, Tensor? lc_tail, Tensor? dout, Tensor? lse, Tensor? delta, Tensor? q2k_ptr, Tensor? q2k_idx, Tensor? bits_a, Tensor? bits_ab, Tensor? blk_cnt, Tensor? add_dq, int add_nb, Tensor? dq_acc, Tensor(a!)? dq, int BH, int L, int D, int RM, int phases) -> ()");
  m.def("vsa_rep_bwd_tables_f16(Tensor? q, Tensor? dout, Tensor? k_tab, Tensor? v_tab, Tensor? lc, int lc_stride, Tensor? lse, Tensor? delta, Tensor? bits_a, Tensor? bits_ab, Tensor(a!)? dk_tab, Tensor(b!)? dv_tab, int BH, int L, int D, int RM, int tier) -> ()");
  m.def("vsa_rep_bwd_both_tables_f16(Tensor? q, Tensor? dout, Tensor? k_mid, Tensor? v_mid, Tensor? lc_mid, int lc_mid_stride, Tensor? k_tail, Tensor? v_tail, Tensor? lc_tail, Tensor? lse, Tensor? delta, Tensor? bits_a, Tensor? bits_ab, Tensor(a!)? dk_mid, Tensor(b!)? dv_mid, Tensor(c!)? dk_tail, Tensor(d!)? dv_tail, int BH, int L, int D, int RM) -> ()");
  m.def("vsa_rep_build_kmeans_f16(Tensor? k, Tensor? v, Tensor? blk_cnt, Tensor(a!)? k_mid, Tensor(b!)? v_mid, Tensor(c!)? lc_mid, Tensor(d!)? counts, Tensor(e!)? labels, int BH, int L, int D, int RM, int iters, int seed) -> ()");
  m.def("vsa_rep_unpool_f16(Tensor? acc_k, Tensor? acc_v, Tensor? dk_mid, Tensor? dv_mid, Tensor? dk_tail, Tensor? dv_tail, Tensor? blk_cnt, Tensor? labels, Tensor? mid_counts, Tensor(a!)? dk, Tensor(b!)? dv, int BH, int L, int D, int RM) -> ()");
  m.def("vsa_row_dot_f16(Tensor? x, Tensor? y, Tensor? blk_cnt, Tensor(a!)? out, int BH, int L, int D) -> ()");
}
TORCH_LIBRARY_IMPL(echosparse_gfx950, CUDA, m) {
  m.impl("es_block_attention", TORCH_FN(op_es_block_attention));
  m.impl("es_sparse_attention", TORCH_FN(op_es_sparse_attention));
  m.impl("es_exact_fallback", TORCH_FN(op_es_exact_fallback));
  m.impl("es_compensate_fallback", TORCH_FN(op_es_compensate_fallback));
  m.impl("es_dense_attention", TORCH_FN(op_es_dense_attention));
  m.impl("es_dense_attention_kv", TORCH_FN(op_es_dense_attention_kv));
  m.impl("es_dense_attention_ws", TORCH_FN(op_es_dense_attention_ws));
  m.impl("es_block_means", TORCH_FN(op_es_block_means));
  m.impl("es_estimate_skipped", TORCH_FN(op_es_estimate_skipped));
  m.impl("es_full_step_scales", TORCH_FN(op_es_full_step_scales));
  m.impl("es_select_blocks", TORCH_FN(op_es_select_blocks));
  m.impl("es_pack_plan", TORCH_FN(op_es_pack_plan));
  m.impl("es_rebuild_plan", TORCH_FN(op_es_rebuild_plan));
  m.impl("es_representatives", TORCH_FN(op_es_representatives));
  m.impl("es_representatives_noalloc", TORCH_FN(op_es_representatives_noalloc));
  m.impl("vsa_pool", TORCH_FN(op_vsa_pool));
  m.impl("vsa_fuse_fwd", TORCH_FN(op_vsa_fuse_fwd));
  m.impl("vsa_fuse_bwd", TORCH_FN(op_vsa_fuse_bwd));
  m.impl("vsa_finalize", TORCH_FN(op_vsa_finalize));
  m.impl("vsa_attn_fwd", TORCH_FN(op_vsa_attn_fwd));
  m.impl("vsa_attn_fwd_tasks", TORCH_FN(op_vsa_attn_fwd_tasks));
  m.impl("vsa_attn_bwd_kv", TORCH_FN(op_vsa_attn_bwd_kv));
  m.impl("vsa_attn_bwd_kv_tasks", TORCH_FN(op_vsa_attn_bwd_kv_tasks));
  m.impl("vsa_attn_bwd_q", TORCH_FN(op_vsa_attn_bwd_q));
  m.impl("vsa_attn_bwd_q_tasks", TORCH_FN(op_vsa_attn_bwd_q_tasks));
  m.impl("vsa_block_scores", TORCH_FN(op_vsa_block_scores));
  m.impl("vsa_route_rows", TORCH_FN(op_vsa_route_rows));
  m.impl("vsa_row_topk", TORCH_FN(op_vsa_row_topk));
  m.impl("vsa_router_lse", TORCH_FN(op_vsa_router_lse));
  m.impl("vsa_router_scores", TORCH_FN(op_vsa_router_scores));
  m.impl("vsa_global_topk", TORCH_FN(op_vsa_global_topk));
  m.impl("vsa_csr_transpose", TORCH_FN(op_vsa_csr_transpose));
  m.impl("vsa_dense_lists", TORCH_FN(op_vsa_dense_lists));
  m.impl("vsa_split_plan", TORCH_FN(op_vsa_split_plan));
  m.impl("vsa_split_merge_fwd", TORCH_FN(op_vsa_split_merge_fwd));
  m.impl("vsa_split_merge_sum", TORCH_FN(op_vsa_split_merge_sum));
  m.impl("vsa_rep_build", TORCH_FN(op_vsa_rep_build));
  m.impl("vsa_rep_build_kmeans", TORCH_FN(op_vsa_rep_build_kmeans));
  m.impl("vsa_row_tiers", TORCH_FN(op_vsa_row_tiers));
  m.impl("vsa_rep_attn_fwd", TORCH_FN(op_vsa_rep_attn_fwd));
  m.impl("vsa_rep_attn_bwd_q", TORCH_FN(op_vsa_rep_attn_bwd_q));
  m.impl("vsa_rep_bwd_tables", TORCH_FN(op_vsa_rep_bwd_tables));
  m.impl("vsa_rep_bwd_both_tables", TORCH_FN(op_vsa_rep_bwd_both_tables));
  m.impl("vsa_rep_unpool", TORCH_FN(op_vsa_rep_unpool));
  m.impl("vsa_row_dot", TORCH_FN(op_vsa_row_dot));
  m.impl("vsa_tier_b_lists", TORCH_FN(op_vsa_tier_b_lists));
  m.impl("vsa_pool_f16", TORCH_FN(op_vsa_pool_f16));
  m.impl("vsa_fuse_fwd_f16", TORCH_FN(op_vsa_fuse_fwd_f16));
  m.impl("vsa_fuse_bwd_f16", TORCH_FN(op_vsa_fuse_bwd_f16));
  m.impl("vsa_finalize_f16", TORCH_FN(op_vsa_finalize_f16));
  m.impl("vsa_attn_fwd_f16", TORCH_FN(op_vsa_attn_fwd_f16));
  m.impl("vsa_attn_fwd_tasks_f16", TORCH_FN(op_vsa_attn_fwd_tasks_f16));
  m.impl("vsa_attn_bwd_kv_f16", TORCH_FN(op_vsa_attn_bwd_kv_f16));
  m.impl("vsa_attn_bwd_kv_tasks_f16", TORCH_FN(op_vsa_attn_bwd_kv_tasks_f16));
  m.impl("vsa_attn_bwd_q_f16", TORCH_FN(op_vsa_attn_bwd_q_f16));
  m.impl("vsa_attn_bwd_q_tasks_f16", TORCH_FN(op_vsa_attn_bwd_q_tasks_f16));
  m.impl("vsa_block_scores_f16", TORCH_FN(op_vsa_block_scores_f16));
  m.impl("vsa_route_rows_f16", TORCH_FN(op_vsa_route_rows_f16));
  m.impl("vsa_row_topk_f16", TORCH_FN(op_vsa_row_topk_f16));
  m.impl("vsa_router_lse_f16", TORCH_FN(op_vsa_router_lse_f16));
  m.impl("vsa_router_scores_f16", TORCH_FN(op_vsa_router_scores_f16));
  m.impl("vsa_split_merge_fwd_f16", TORCH_FN(op_vsa_split_merge_fwd_f16));
  m.impl("vsa_split_merge_sum_f16", TORCH_FN(op_vsa_split_merge_sum_f16));
  m.impl("vsa_rep_build_f16", TORCH_FN(op_vsa_rep_build_f16));
  m.impl("vsa_rep_attn_fwd_f16", TORCH_FN(op_vsa_rep_attn_fwd_f16));
  m.impl("vsa_rep_attn_bwd_q_f16", TORCH_FN(op_vsa_rep_attn_bwd_q_f16));
  m.impl("vsa_rep_bwd_tables_f16", TORCH_FN(op_vsa_rep_bwd_tables_f16));
  m.impl("vsa_rep_bwd_both_tables_f16", TORCH_FN(op_vsa_rep_bwd_both_tables_f16));
  m.impl("vsa_rep_build_kmeans_f16", TORCH_FN(op_vsa_rep_build_kmeans_f16));
  m.impl("vsa_rep_unpool_f16", TORCH_FN(op_vsa_rep_unpool_f16));
  m.impl("vsa_row_dot_f16", TORCH_FN(op_vsa_row_dot_f16));
}
TORCH_LIBRARY_IMPL(echosparse_gfx950, CPU, m) {
  m.impl("es_block_attention", TORCH_FN(op_es_block_attention));
  m.impl("es_sparse_attention", TORCH_FN(op_es_sparse_attention));
  m.impl("es_exact_fallback", TORCH_FN(op_es_exact_fallback));
  m.impl("es_compensate_fallback", TORCH_FN(op_es_compensate_fallback));
  m.impl("es_dense_attention", TORCH_FN(op_es_dense_attention));
  m.impl("es_dense_attention_kv", TORCH_FN(op_es_dense_attention_kv));
  m.impl("es_dense_attention_ws", TORCH_FN(op_es_dense_attention_ws));
  m.impl("es_block_means", TORCH_FN(op_es_block_means));
  m.impl("es_estimate_skipped", TORCH_FN(op_es_estimate_skipped));
  m.impl("es_full_step_scales", TORCH_FN(op_es_full_step_scales));
  m.impl("es_select_blocks", TORCH_FN(op_es_select_blocks));
  m.impl("es_pack_plan", TORCH_FN(op_es_pack_plan));
  m.impl("es_rebuild_plan", TORCH_FN(op_es_rebuild_plan));
  m.impl("es_representatives", TORCH_FN(op_es_representatives));
  m.impl("es_representatives_noalloc", TORCH_FN(op_es_representatives_noalloc));
  m.impl("vsa_pool", TORCH_FN(op_vsa_pool));
  m.impl("vsa_fuse_fwd", TORCH_FN(op_vsa_fuse_fwd));
  m.impl("vsa_fuse_bwd", TORCH_FN(op_vsa_fuse_bwd));
  m.impl("vsa_finalize", TORCH_FN(op_vsa_finalize));
  m.impl("vsa_attn_fwd", TORCH_FN(op_vsa_attn_fwd));
  m.impl("vsa_attn_fwd_tasks", TORCH_FN(op_vsa_attn_fwd_tasks));
  m.impl("vsa_attn_bwd_kv", TORCH_FN(op_vsa_attn_bwd_kv));
  m.impl("vsa_attn_bwd_kv_tasks", TORCH_FN(op_vsa_attn_bwd_kv_tasks));
  m.impl("vsa_attn_bwd_q", TORCH_FN(op_vsa_attn_bwd_q));
  m.impl("vsa_attn_bwd_q_tasks", TORCH_FN(op_vsa_attn_bwd_q_tasks));
  m.impl("vsa_block_scores", TORCH_FN(op_vsa_block_scores));
  m.impl("vsa_route_rows", TORCH_FN(op_vsa_route_rows));
  m.impl("vsa_row_topk", TORCH_FN(op_vsa_row_topk));
  m.impl("vsa_router_lse", TORCH_FN(op_vsa_router_lse));
  m.impl("vsa_router_scores", TORCH_FN(op_vsa_router_scores));
  m.impl("vsa_global_topk", TORCH_FN(op_vsa_global_topk));
  m.impl("vsa_csr_transpose", TORCH_FN(op_vsa_csr_transpose));
  m.impl("vsa_dense_lists", TORCH_FN(op_vsa_dense_lists));
  m.impl("vsa_split_plan", TORCH_FN(op_vsa_split_plan));
  m.impl("vsa_split_merge_fwd", TORCH_FN(op_vsa_split_merge_fwd));
  m.impl("vsa_split_merge_sum", TORCH_FN(op_vsa_split_merge_sum));
  m.impl("vsa_rep_build", TORCH_FN(op_vsa_rep_build));
  m.impl("vsa_rep_build_kmeans", TORCH_FN(op_vsa_rep_build_kmeans));
  m.impl("vsa_row_tiers", TORCH_FN(op_vsa_row_tiers));
  m.impl("vsa_rep_attn_fwd", TORCH_FN(op_vsa_rep_attn_fwd));
  m.impl("vsa_rep_attn_bwd_q", TORCH_FN(op_vsa_rep_attn_bwd_q));
  m.impl("vsa_rep_bwd_tables", TORCH_FN(op_vsa_rep_bwd_tables));
  m.impl("vsa_rep_bwd_both_tables", TORCH_FN(op_vsa_rep_bwd_both_tables));
  m.impl("vsa_rep_unpool", TORCH_FN(op_vsa_rep_unpool));
  m.impl("vsa_row_dot", TORCH_FN(op_vsa_row_dot));
  m.impl("vsa_tier_b_lists", TORCH_FN(op_vsa_tier_b_lists));
  m.impl("vsa_pool_f16", TORCH_FN(op_vsa_pool_f16));
  m.impl("vsa_fuse_fwd_f16", TORCH_FN(op_vsa_fuse_fwd_f16));
  m.impl("vsa_fuse_bwd_f16", TORCH_FN(op_vsa_fuse_bwd_f16));
  m.impl("vsa_finalize_f16", TORCH_FN(op_vsa_finalize_f16));
  m.impl("vsa_attn_fwd_f16", TORCH_FN(op_vsa_attn_fwd_f16));
  m.impl("vsa_attn_fwd_tasks_f16", TORCH_FN(op_vsa_attn_fwd_tasks_f16));
  m.impl("vsa_attn_bwd_kv_f16", TORCH_FN(op_vsa_attn_bwd_kv_f16));
  m.impl("vsa_attn_bwd_kv_tasks_f16", TORCH_FN(op_vsa_attn_bwd_kv_tasks_f16));
  m.impl("vsa_attn_bwd_q_f16", TORCH_FN(op_vsa_attn_bwd_q_f16));
  m.impl("vsa_attn_bwd_q_tasks_f16", TORCH_FN(op_vsa_attn_bwd_q_tasks_f16));
  m.impl("vsa_block_scores_f16", TORCH_FN(op_vsa_block_scores_f16));
  m.impl("vsa_route_rows_f16", TORCH_FN(op_vsa_route_rows_f16));
  m.impl("vsa_row_topk_f16", TORCH_FN(op_vsa_row_topk_f16));
  m.impl("vsa_router_lse_f16", TORCH_FN(op_vsa_router_lse_f16));
  m.impl("vsa_router_scores_f16", TORCH_FN(op_vsa_router_scores_f16));
  m.impl("vsa_split_merge_fwd_f16", TORCH_FN(op_vsa_split_merge_fwd_f16));
  m.impl("vsa_split_merge_sum_f16", TORCH_FN(op_vsa_split_merge_sum_f16));
  m.impl("vsa_rep_build_f16", TORCH_FN(op_vsa_rep_build_f16));
  m.impl("vsa_rep_attn_fwd_f16", TORCH_FN(op_vsa_rep_attn_fwd_f16));
  m.impl("vsa_rep_attn_bwd_q_f16", TORCH_FN(op_vsa_rep_attn_bwd_q_f16));
  m.impl("vsa_rep_bwd_tables_f16", TORCH_FN(op_vsa_rep_bwd_tables_f16));
  m.impl("vsa_rep_bwd_both_tables_f16", TORCH_FN(op_vsa_rep_bwd_both_tables_f16));
  m.impl("vsa_rep_build_kmeans_f16", TORCH_FN(op_vsa_rep_build_kmeans_f16));
  m.impl("vsa_rep_unpool_f16", TORCH_FN(op_vsa_rep_unpool_f16));
  m.impl("vsa_row_dot_f16", TORCH_FN(op_vsa_row_dot_f16));
}
TORCH_LIBRARY_IMPL(echosparse_gfx950, Meta, m) {
  m.impl("es_block_attention", TORCH_FN(meta_es_block_attention));
  m.impl("es_sparse_attention", TORCH_FN(meta_es_sparse_attention));
  m.impl("es_exact_fallback", TORCH_FN(meta_es_exact_fallback));
  m.impl("es_compensate_fallback", TORCH_FN(meta_es_compensate_fallback));
  m.impl("es_dense_attention", TORCH_FN(meta_es_dense_attention));
  m.impl("es_dense_attention_kv", TORCH_FN(meta_es_dense_attention_kv));
  m.impl("es_dense_attention_ws", TORCH_FN(meta_es_dense_attention_ws));
  m.impl("es_block_means", TORCH_FN(meta_es_block_means));
  m.impl("es_estimate_skipped", TORCH_FN(meta_es_estimate_skipped));
  m.impl("es_full_step_scales", TORCH_FN(meta_es_full_step_scales));
  m.impl("es_select_blocks", TORCH_FN(meta_es_select_blocks));
  m.impl("es_pack_plan", TORCH_FN(meta_es_pack_plan));
  m.impl("es_rebuild_plan", TORCH_FN(meta_es_rebuild_plan));
  m.impl("es_representatives", TORCH_FN(meta_es_representatives));
  m.impl("es_representatives_noalloc", TORCH_FN(meta_es_representatives_noalloc));
  m.impl("vsa_pool", TORCH_FN(meta_vsa_pool));
  m.impl("vsa_fuse_fwd", TORCH_FN(meta_vsa_fuse_fwd));
  m.impl("vsa_fuse_bwd", TORCH_FN(meta_vsa_fuse_bwd));
  m.impl("vsa_finalize", TORCH_FN(meta_vsa_finalize));
  m.impl("vsa_attn_fwd", TORCH_FN(meta_vsa_attn_fwd));
  m.impl("vsa_attn_fwd_tasks", TORCH_FN(meta_vsa_attn_fwd_tasks));
  m.impl("vsa_attn_bwd_kv", TORCH_FN(meta_vsa_attn_bwd_kv));
  m.impl("vsa_attn_bwd_kv_tasks", TORCH_FN(meta_vsa_attn_bwd_kv_tasks));
  m.impl("vsa_attn_bwd_q", TORCH_FN(meta_vsa_attn_bwd_q));
  m.impl("vsa_attn_bwd_q_tasks", TORCH_FN(meta_vsa_attn_bwd_q_tasks));
  m.impl("vsa_block_scores", TORCH_FN(meta_vsa_block_scores));
  m.impl("vsa_route_rows", TORCH_FN(meta_vsa_route_rows));
  m.impl("vsa_row_topk", TORCH_FN(meta_vsa_row_topk));
  m.impl("vsa_router_lse", TORCH_FN(meta_vsa_router_lse));
  m.impl("vsa_router_scores", TORCH_FN(meta_vsa_router_scores));
  m.impl("vsa_global_topk", TORCH_FN(meta_vsa_global_topk));
  m.impl("vsa_csr_transpose", TORCH_FN(meta_vsa_csr_transpose));
  m.impl("vsa_dense_lists", TORCH_FN(meta_vsa_dense_lists));
  m.impl("vsa_split_plan", TORCH_FN(meta_vsa_split_plan));
  m.impl("vsa_split_merge_fwd", TORCH_FN(meta_vsa_split_merge_fwd));
  m.impl("vsa_split_merge_sum", TORCH_FN(meta_vsa_split_merge_sum));
  m.impl("vsa_rep_build", TORCH_FN(meta_vsa_rep_build));
  m.impl("vsa_rep_build_kmeans", TORCH_FN(meta_vsa_rep_build_kmeans));
  m.impl("vsa_row_tiers", TORCH_FN(meta_vsa_row_tiers));
  m.impl("vsa_rep_attn_fwd", TORCH_FN(meta_vsa_rep_attn_fwd));
  m.impl("vsa_rep_attn_bwd_q", TORCH_FN(meta_vsa_rep_attn_bwd_q));
  m.impl("vsa_rep_bwd_tables", TORCH_FN(meta_vsa_rep_bwd_tables));
  m.impl("vsa_rep_bwd_both_tables", TORCH_FN(meta_vsa_rep_bwd_both_tables));
  m.impl("vsa_rep_unpool", TORCH_FN(meta_vsa_rep_unpool));
  m.impl("vsa_row_dot", TORCH_FN(meta_vsa_row_dot));
  m.impl("vsa_tier_b_lists", TORCH_FN(meta_vsa_tier_b_lists));
  m.impl("vsa_pool_f16", TORCH_FN(meta_vsa_pool_f16));
  m.impl("vsa_fuse_fwd_f16", TORCH_FN(meta_vsa_fuse_fwd_f16));
  m.impl("vsa_fuse_bwd_f16", TORCH_FN(meta_vsa_fuse_bwd_f16));
  m.impl("vsa_finalize_f16", TORCH_FN(meta_vsa_finalize_f16));
  m.impl("vsa_attn_fwd_f16", TORCH_FN(meta_vsa_attn_fwd_f16));
  m.impl("vsa_attn_fwd_tasks_f16", TORCH_FN(meta_vsa_attn_fwd_tasks_f16));
  m.impl("vsa_attn_bwd_kv_f16", TORCH_FN(meta_vsa_attn_bwd_kv_f16));
  m.impl("vsa_attn_bwd_kv_tasks_f16", TORCH_FN(meta_vsa_attn_bwd_kv_tasks_f16));
  m.impl("vsa_attn_bwd_q_f16", TORCH_FN(meta_vsa_attn_bwd_q_f16));
  m.impl("vsa_attn_bwd_q_tasks_f16", TORCH_FN(meta_vsa_attn_bwd_q_tasks_f16));
  m.impl("vsa_block_scores_f16", TORCH_FN(meta_vsa_block_scores_f16));
  m.impl("vsa_route_rows_f16", TORCH_FN(meta_vsa_route_rows_f16));
  m.impl("vsa_row_topk_f16", TORCH_FN(meta_vsa_row_topk_f16));
  m.impl("vsa_router_lse_f16", TORCH_FN(meta_vsa_router_lse_f16));
  m.impl("vsa_router_scores_f16", TORCH_FN(meta_vsa_router_scores_f16));
  m.impl("vsa_split_merge_fwd_f16", TORCH_FN(meta_vsa_split_merge_fwd_f16));
  m.impl("vsa_split_merge_sum_f16", TORCH_FN(meta_vsa_split_merge_sum_f16));
  m.impl("vsa_rep_build_f16", TORCH_FN(meta_vsa_rep_build_f16));
  m.impl("vsa_rep_attn_fwd_f16", TORCH_FN(meta_vsa_rep_attn_fwd_f16));
  m.impl("vsa_rep_attn_bwd_q_f16", TORCH_FN(meta_vsa_rep_attn_bwd_q_f16));
  m.impl("vsa_rep_bwd_tables_f16", TORCH_FN(meta_vsa_rep_bwd_tables_f16));
  m.impl("vsa_rep_bwd_both_tables_f16", TORCH_FN(meta_vsa_rep_bwd_both_tables_f16));
  m.impl("vsa_rep_build_kmeans_f16", TORCH_FN(meta_vsa_rep_build_kmeans_f16));
  m.impl("vsa_rep_unpool_f16", TORCH_FN(meta_vsa_rep_unpool_f16));
  m.impl("vsa_row_dot_f16", TORCH_FN(meta_vsa_row_dot_f16));
}
