// torch.ops.fxpr.* on the GPU: the launchers of fxpr_vllm/_kernels/*.py as
// native kernels of the "CUDA" dispatch key (which PyTorch-ROCm's tensors use).
//
// Same validation order, error classes (ValueError / TypeError / RuntimeError),
// contiguity rules, empty-tensor returns, allocations and C entry points as
// those launchers, which stay the callable form with explicit split counts. A
// decode step runs a dozen of these calls a layer: as Python functions behind
// the dispatcher each cost 9-20 us of host time (argument checks, torch calls
// and a ctypes call of up to 40 arguments), more than the kernels they launch.
// One-row 4096 x 4096 linear: 12.6 -> 8.3 us a call; attention over 4 prompts of
// up to 36 tokens: 20.0 -> 10.5 us; the four calls of a small encode / sum /
// decode chain: 37.4 -> 20.9 us.
// Compiled by the host compiler against torch's headers; links libfxpr_hip.so.

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <cmath>
#include <cstdint>
#include <optional>
#include <tuple>

#include "fxpr.h"

namespace {

using at::Tensor;

int code_of(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return FXPR_DTYPE_F16;
    case at::kBFloat16: return FXPR_DTYPE_BF16;
    case at::kFloat: return FXPR_DTYPE_F32;
    case at::kDouble: return FXPR_DTYPE_F64;
    case at::kShort: return FXPR_DTYPE_I16;
    case at::kInt: return FXPR_DTYPE_I32;
    case at::kLong: return FXPR_DTYPE_I64;
    default: return -1;
  }
}

bool is_io(at::ScalarType t) { return t == at::kFloat || t == at::kHalf || t == at::kBFloat16; }

at::ScalarType int_type(int64_t bits) { return bits == 16 ? at::kShort : bits == 32 ? at::kInt : at::kLong; }

void check_int_bits(int64_t n) { TORCH_CHECK_VALUE(n == 16 || n == 32 || n == 64, "int_bits must be 16/32/64, got ", n); }

void check_frac_bits(int64_t n) {
  TORCH_CHECK_VALUE(n == 8 || n == 16 || n == 32, "fxp_frac_bits must be 8/16/32, got ", n);
}

void check_rc(int rc, const char* name) {
  TORCH_CHECK(rc == 0, name, " failed: ", fxpr_error_string(rc), " (code ", rc, ")");
}

void* stream_of(const Tensor& t) {
  return static_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

Tensor bytes(int64_t n, const Tensor& like) { return at::empty({n}, like.options().dtype(at::kByte)); }

Tensor as_2d(const Tensor& x) { return x.reshape({-1, x.size(-1)}); }

Tensor float_to_fixed(const Tensor& x, int64_t int_bits, int64_t frac_bits) {
  check_int_bits(int_bits);
  check_frac_bits(frac_bits);
  TORCH_CHECK(x.is_cuda(), "float_to_fixed: input must be CUDA");
  const auto t = x.scalar_type();
  TORCH_CHECK_TYPE(t == at::kHalf || t == at::kFloat || t == at::kDouble, "float_to_fixed: unsupported input dtype ", t,
                   "; expected float16, float32 or float64");
  const c10::DeviceGuard guard(x.device());
  const Tensor xc = x.contiguous();
  Tensor y = at::empty(xc.sizes(), xc.options().dtype(int_type(int_bits)));
  if (xc.numel() == 0) return y;
  check_rc(fxpr_float_to_fixed(xc.const_data_ptr(), code_of(t), y.mutable_data_ptr(), int(int_bits), int(frac_bits),
                               xc.numel(), stream_of(xc)),
           "fxpr_float_to_fixed");
  return y;
}

Tensor fixed_to_float(const Tensor& x, int64_t float_bits, int64_t frac_bits) {
  TORCH_CHECK_VALUE(float_bits == 16 || float_bits == 32 || float_bits == 64, "float_bits must be 16/32/64, got ",
                    float_bits);
  check_frac_bits(frac_bits);
  TORCH_CHECK(x.is_cuda(), "fixed_to_float: input must be CUDA");
  const auto t = x.scalar_type();
  TORCH_CHECK_TYPE(t == at::kShort || t == at::kInt || t == at::kLong, "fixed_to_float: unsupported input dtype ", t,
                   "; expected int16, int32 or int64");
  const c10::DeviceGuard guard(x.device());
  const Tensor xc = x.contiguous();
  const auto out = float_bits == 16 ? at::kHalf : float_bits == 32 ? at::kFloat : at::kDouble;
  Tensor y = at::empty(xc.sizes(), xc.options().dtype(out));
  if (xc.numel() == 0) return y;
  check_rc(fxpr_fixed_to_float(xc.const_data_ptr(), code_of(t), y.mutable_data_ptr(), int(float_bits), int(frac_bits),
                               xc.numel(), stream_of(xc)),
           "fxpr_fixed_to_float");
  return y;
}

Tensor fixed_row_sum(const Tensor& q, int64_t int_bits) {
  check_int_bits(int_bits);
  TORCH_CHECK(q.is_cuda(), "fixed_row_sum: input must be CUDA");
  const auto t = q.scalar_type();
  TORCH_CHECK_TYPE(t == at::kShort || t == at::kInt || t == at::kLong, "fixed_row_sum: unsupported input dtype ", t,
                   "; expected int16, int32 or int64");
  const c10::DeviceGuard guard(q.device());
  const Tensor qc = q.contiguous();
  const auto shape = qc.dim() ? qc.sizes().slice(0, qc.dim() - 1) : at::IntArrayRef{};
  const int64_t cols = qc.dim() ? qc.size(-1) : 1;
  Tensor out = at::empty(shape, qc.options().dtype(int_type(int_bits)));
  if (out.numel() == 0) return out;
  if (cols == 0) return out.zero_();
  check_rc(fxpr_fixed_row_sum(qc.const_data_ptr(), code_of(t), out.mutable_data_ptr(), int(int_bits), out.numel(), cols,
                              stream_of(qc)),
           "fxpr_fixed_row_sum");
  return out;
}

Tensor rms_norm_impl(const Tensor& x, const Tensor* residual, const Tensor& w, double eps) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda(), "rms_norm: x and w must be CUDA");
  const auto t = x.scalar_type();
  TORCH_CHECK_TYPE(is_io(t), "rms_norm: unsupported input dtype ", t, "; expected float32, float16 or bfloat16");
  TORCH_CHECK_TYPE(w.scalar_type() == t, "rms_norm: weight dtype must match input dtype");
  if (residual) {
    TORCH_CHECK(residual->is_cuda(), "rms_norm: residual must be CUDA");
    TORCH_CHECK_TYPE(residual->scalar_type() == t, "rms_norm: residual dtype must match input dtype");
    TORCH_CHECK_VALUE(residual->sizes() == x.sizes(), "rms_norm: residual shape must match x");
  }
  const c10::DeviceGuard guard(x.device());
  const Tensor x2 = as_2d(x).contiguous();
  Tensor y = at::empty(x2.sizes(), x2.options());
  Tensor r2;
  if (residual) r2 = as_2d(*residual).contiguous();
  const int64_t rows = x2.size(0), hidden = x2.size(1);
  auto copy_back = [&]() {
    if (residual && r2.const_data_ptr() != residual->const_data_ptr()) residual->copy_(r2.view_as(*residual));
  };
  if (rows == 0 || hidden == 0) {
    copy_back();
    return y.view_as(x);
  }
  TORCH_CHECK_VALUE(w.numel() == hidden, "rms_norm: weight has ", w.numel(), " elements, hidden size is ", hidden);
  const Tensor wc = w.contiguous();
  check_rc(fxpr_rms_norm(x2.const_data_ptr(), residual ? r2.mutable_data_ptr() : nullptr, wc.const_data_ptr(),
                         y.mutable_data_ptr(), code_of(t), rows, hidden, float(eps), stream_of(x2)),
           "fxpr_rms_norm");
  copy_back();
  return y.view_as(x);
}

Tensor rms_norm(const Tensor& x, const Tensor& w, double eps) { return rms_norm_impl(x, nullptr, w, eps); }

Tensor rms_norm_residual(const Tensor& x, Tensor& residual, const Tensor& w, double eps) {
  return rms_norm_impl(x, &residual, w, eps);
}

Tensor log_softmax(const Tensor& x, int64_t int_bits, int64_t frac_bits, std::optional<at::ScalarType> out_dtype) {
  check_int_bits(int_bits);
  check_frac_bits(frac_bits);
  TORCH_CHECK(x.is_cuda(), "log_softmax_fxp: input must be CUDA");
  const auto t = x.scalar_type(), ot = out_dtype.value_or(t);
  TORCH_CHECK_TYPE(is_io(t), "log_softmax_fxp: unsupported input dtype ", t, "; expected float32, float16 or bfloat16");
  TORCH_CHECK_TYPE(ot == t || ot == at::kFloat, "log_softmax_fxp: output dtype must be ", t, " or float32, got ", ot);
  const c10::DeviceGuard guard(x.device());
  const Tensor x2 = x.dim() > 0 ? as_2d(x).contiguous() : x.reshape({1, 1});
  Tensor y = at::empty(x2.sizes(), x2.options().dtype(ot));
  if (x2.size(0) && x2.size(1))
    check_rc(fxpr_log_softmax(x2.const_data_ptr(), code_of(t), y.mutable_data_ptr(), code_of(ot), x2.size(0), x2.size(1),
                              int(int_bits), int(frac_bits), stream_of(x2)),
             "fxpr_log_softmax");
  return y.view(x.sizes());
}

std::tuple<Tensor, Tensor, Tensor, Tensor> sample_greedy(const Tensor& logits, int64_t k, int64_t int_bits,
                                                         int64_t frac_bits) {
  constexpr int64_t kMaxLogprobs = 64;
  check_int_bits(int_bits);
  check_frac_bits(frac_bits);
  TORCH_CHECK(logits.is_cuda(), "sample_greedy_fxp: logits must be CUDA");
  const auto t = logits.scalar_type();
  TORCH_CHECK_TYPE(is_io(t), "sample_greedy_fxp: unsupported dtype ", t, "; expected float32, float16 or bfloat16");
  TORCH_CHECK_VALUE(logits.dim() > 0, "sample_greedy_fxp: logits need a vocabulary dimension");
  const int64_t vocab = logits.size(-1), most = std::min(kMaxLogprobs, vocab);
  TORCH_CHECK_VALUE(vocab > 0, "sample_greedy_fxp: empty vocabulary");
  TORCH_CHECK_VALUE(0 <= k && k <= most, "sample_greedy_fxp: num_logprobs must be in [0, ", most, "], got ", k);
  const c10::DeviceGuard guard(logits.device());
  const Tensor x = logits.reshape({-1, vocab}).contiguous();
  const int64_t rows = x.size(0);
  Tensor ids = at::empty({rows}, x.options().dtype(at::kLong)), lp = at::empty({rows}, x.options().dtype(at::kFloat));
  Tensor top = at::empty({rows, k}, x.options().dtype(at::kLong));
  Tensor top_lp = at::empty({rows, k}, x.options().dtype(at::kFloat));
  if (rows) {
    // few rows: the library spreads each row over several workgroups, its
    // partials in this workspace (caching allocator: capture-safe)
    const int64_t n = fxpr_sample_greedy_workspace_bytes(rows, int(k));
    Tensor ws = n > 0 ? bytes(n, x) : Tensor();
    check_rc(fxpr_sample_greedy(x.const_data_ptr(), code_of(t), rows, vocab, int(k), int(int_bits), int(frac_bits),
                                ids.mutable_data_ptr<int64_t>(), lp.mutable_data_ptr<float>(),
                                k ? top.mutable_data_ptr<int64_t>() : nullptr, k ? top_lp.mutable_data_ptr<float>() : nullptr,
                                n > 0 ? ws.mutable_data_ptr() : nullptr, n, stream_of(x)),
             "fxpr_sample_greedy");
  }
  const auto lead = logits.sizes().slice(0, logits.dim() - 1);
  auto with_k = lead.vec();
  with_k.push_back(k);
  return {ids.view(lead), lp.view(lead), top.view(with_k), top_lp.view(with_k)};
}

Tensor gemm(const Tensor& a_in, const Tensor& b_in, const std::optional<Tensor>& bias, int64_t int_bits,
            int64_t frac_bits) {
  check_int_bits(int_bits);
  check_frac_bits(frac_bits);
  TORCH_CHECK(a_in.is_cuda() && b_in.is_cuda(), "gemm_fxp: a and b must be CUDA");
  const auto t = a_in.scalar_type();
  TORCH_CHECK_TYPE(is_io(t), "gemm_fxp: unsupported dtype ", t, "; expected float16, bfloat16 or float32");
  TORCH_CHECK_TYPE(b_in.scalar_type() == t, "gemm_fxp: a and b must share a dtype");
  TORCH_CHECK_VALUE(a_in.dim() == 2 && b_in.dim() == 2 && a_in.size(1) == b_in.size(0), "gemm_fxp: shape mismatch ",
                    a_in.sizes(), " x ", b_in.sizes());
  const c10::DeviceGuard guard(a_in.device());
  const int64_t M = a_in.size(0), K = a_in.size(1), N = b_in.size(1);
  Tensor c = at::empty({M, N}, a_in.options());
  if (M == 0 || N == 0) return c;
  const Tensor a = a_in.stride(1) != 1 && K > 1 ? a_in.contiguous() : a_in;
  const Tensor b = b_in.stride(0) != 1 && b_in.stride(1) != 1 ? b_in.contiguous() : b_in;
  Tensor bias32;
  if (bias.has_value() && bias->defined()) {
    TORCH_CHECK_VALUE(bias->numel() == N, "gemm_fxp: bias has ", bias->numel(), " elements, expected ", N);
    bias32 = bias->reshape({N}).to(at::kFloat).contiguous();
  }
  const int code = code_of(t), bits = int(int_bits);
  const int split_k =
      fxpr_gemm_layout_splits(M, N, K, code, bits, int(frac_bits), a.stride(0), b.stride(0), b.stride(1));
  const int64_t n = fxpr_gemm_workspace_bytes(M, N, K, code, bits, split_k);
  Tensor ws = n > 0 ? bytes(n, a) : Tensor();
  check_rc(fxpr_gemm(a.const_data_ptr(), b.const_data_ptr(), bias32.defined() ? bias32.const_data_ptr<float>() : nullptr,
                     c.mutable_data_ptr(), code, M, N, K, a.stride(0), a.stride(1), b.stride(0), b.stride(1), c.stride(0),
                     c.stride(1), bits, int(frac_bits), split_k, n > 0 ? ws.mutable_data_ptr() : nullptr, n,
                     stream_of(a)),
           "fxpr_gemm");
  return c;
}

void unified_attention(const Tensor& q_in, const Tensor& kv_cache, Tensor& o, const Tensor& query_start_loc,
                       const Tensor& seq_lens, const Tensor& block_table, int64_t max_query_len,
                       const std::optional<Tensor>& alibi_slopes, bool is_causal, std::optional<double> softmax_scale,
                       int64_t int_bits, int64_t frac_bits, double logit_softcap, int64_t window_size,
                       int64_t num_kv_splits) {
  check_int_bits(int_bits);
  check_frac_bits(frac_bits);
  TORCH_CHECK(q_in.is_cuda() && kv_cache.is_cuda() && o.is_cuda(), "unified_attention_fxp: tensors must be CUDA");
  const auto t = q_in.scalar_type();
  TORCH_CHECK_TYPE(is_io(t), "unified_attention_fxp: unsupported q dtype ", t);
  TORCH_CHECK_VALUE(kv_cache.dim() == 5 && kv_cache.size(1) == 2,
                    "kv_cache must be (num_blocks, 2, page_size, num_kv_heads, head_dim)");
  TORCH_CHECK_TYPE(kv_cache.scalar_type() == t && o.scalar_type() == t, "kv_cache and o must share dtype with q");
  TORCH_CHECK_TYPE(query_start_loc.scalar_type() == at::kInt, "query_start_loc must be int32");
  TORCH_CHECK_TYPE(seq_lens.scalar_type() == at::kInt, "seq_lens must be int32");
  TORCH_CHECK_TYPE(block_table.scalar_type() == at::kInt, "block_table must be int32");
  TORCH_CHECK_VALUE(num_kv_splits >= 0, "num_kv_splits must be >= 0, got ", num_kv_splits);
  const bool has_alibi = alibi_slopes.has_value() && alibi_slopes->defined() && alibi_slopes->numel() > 0;
  TORCH_CHECK_TYPE(!has_alibi || alibi_slopes->scalar_type() == at::kFloat, "alibi_slopes must be float32");

  const c10::DeviceGuard guard(q_in.device());
  const Tensor k_cache = kv_cache.select(1, 0), v_cache = kv_cache.select(1, 1);
  TORCH_CHECK_VALUE(q_in.dim() == 3, "q must be (num_tokens, num_heads, head_dim)");
  const int64_t num_tokens = q_in.size(0), num_heads = q_in.size(1), head_dim = q_in.size(2);
  const int64_t num_blocks = k_cache.size(0), page_size = k_cache.size(1), num_kv_heads = k_cache.size(2);
  const int64_t num_requests = seq_lens.size(0);
  // (a head count of 0 divides nothing; as Python's modulo)
  TORCH_CHECK(num_kv_heads != 0, "unified_attention_fxp: num_kv_heads must not be 0");
  TORCH_CHECK_VALUE(num_heads % num_kv_heads == 0, "num_heads must be divisible by num_kv_heads");
  TORCH_CHECK_VALUE(k_cache.size(3) == head_dim && o.sizes() == q_in.sizes(), "q, o and kv_cache head sizes must agree");
  if (num_requests == 0 || num_tokens == 0) return;
  const Tensor q = q_in.stride(2) != 1 ? q_in.contiguous() : q_in;
  TORCH_CHECK_VALUE(k_cache.stride(3) == 1, "kv_cache must be contiguous along head_dim");
  Tensor out = o.stride(2) == 1 ? o : at::empty(o.sizes(), o.options());
  Tensor bt = block_table.dim() == 2 ? block_table : block_table.reshape({num_requests, -1});
  if (bt.stride(1) != 1) bt = bt.contiguous();
  const Tensor qsl = query_start_loc.contiguous(), sl = seq_lens.contiguous();
  const Tensor alibi = has_alibi ? alibi_slopes->contiguous() : Tensor();

  constexpr double kRcpLn2 = 1.4426950408889634;
  const double scale = softmax_scale.has_value() ? *softmax_scale : 1.0 / std::sqrt(double(head_dim));
  const float scale_log2 = float(scale * kRcpLn2);
  const float softcap_log2 = logit_softcap > 0.0 ? float(logit_softcap * kRcpLn2) : 0.0f;
  const int64_t max_blocks = bt.size(1);
  const int64_t window = std::max<int64_t>(0, window_size);
  const int64_t n = fxpr_attention_plan(code_of(t), int(num_requests), num_tokens, int(num_heads), int(num_kv_heads),
                                        int(head_dim), int(page_size), int(max_query_len), int(max_blocks),
                                        k_cache.stride(1), v_cache.stride(1), is_causal ? 1 : 0, int(window), int(int_bits),
                                        int(num_kv_splits), nullptr);
  Tensor ws = n > 0 ? bytes(n, q) : Tensor();
  check_rc(fxpr_unified_attention(
               q.const_data_ptr(), k_cache.const_data_ptr(), v_cache.const_data_ptr(), out.mutable_data_ptr(), code_of(t),
               qsl.const_data_ptr<int32_t>(), sl.const_data_ptr<int32_t>(), bt.const_data_ptr<int32_t>(),
               has_alibi ? alibi.const_data_ptr<float>() : nullptr, int(num_requests), num_tokens, int(num_heads),
               int(num_kv_heads), int(head_dim), int(page_size), int(max_query_len), int(max_blocks), num_blocks,
               q.stride(0), q.stride(1), k_cache.stride(0), k_cache.stride(1), k_cache.stride(2), v_cache.stride(0),
               v_cache.stride(1), v_cache.stride(2), out.stride(0), out.stride(1), bt.stride(0), is_causal ? 1 : 0,
               scale_log2, softcap_log2, int(window), int(int_bits), int(frac_bits), int(num_kv_splits),
               n > 0 ? ws.mutable_data_ptr() : nullptr, n, stream_of(q)),
           "fxpr_unified_attention");
  if (!out.is_same(o)) o.copy_(out);
}

void reshape_and_cache(const Tensor& key_in, const Tensor& value_in, Tensor& kv_cache, const Tensor& slot_mapping) {
  TORCH_CHECK(key_in.is_cuda() && value_in.is_cuda() && kv_cache.is_cuda() && slot_mapping.is_cuda(),
              "reshape_and_cache: tensors must be CUDA");
  TORCH_CHECK_VALUE(kv_cache.dim() == 5 && kv_cache.size(1) == 2,
                    "kv_cache must be (num_blocks, 2, block_size, num_kv_heads, head_size)");
  const auto t = kv_cache.scalar_type();
  TORCH_CHECK_TYPE(is_io(t), "reshape_and_cache: unsupported cache dtype ", t);
  TORCH_CHECK_TYPE(key_in.scalar_type() == t && value_in.scalar_type() == t, "key, value and kv_cache must share a dtype");
  const c10::DeviceGuard guard(kv_cache.device());
  const int64_t num_blocks = kv_cache.size(0), block = kv_cache.size(2), heads = kv_cache.size(3), d = kv_cache.size(4);
  Tensor key = key_in.dim() == 2 ? key_in.view({key_in.size(0), heads, d}) : key_in;
  Tensor value = value_in.dim() == 2 ? value_in.view({value_in.size(0), heads, d}) : value_in;
  TORCH_CHECK_VALUE(key.sizes() == value.sizes() && key.dim() == 3 && key.size(1) == heads && key.size(2) == d,
                    "key / value must be [num_tokens, num_kv_heads, head_size] matching the cache");
  const int64_t num_tokens = key.size(0);
  TORCH_CHECK_VALUE(slot_mapping.dim() == 1 && slot_mapping.size(0) >= num_tokens,
                    "slot_mapping must be 1-D with one slot per token");
  if (num_tokens == 0) return;
  if (key.stride(2) != 1) key = key.contiguous();
  if (value.stride(2) != 1) value = value.contiguous();
  const Tensor slots = slot_mapping.to(at::kLong).contiguous();
  const Tensor k_cache = kv_cache.select(1, 0), v_cache = kv_cache.select(1, 1);
  TORCH_CHECK_VALUE(k_cache.stride(3) == 1, "kv_cache must be contiguous along head_size");
  check_rc(fxpr_reshape_and_cache(key.const_data_ptr(), value.const_data_ptr(), k_cache.mutable_data_ptr(),
                                  v_cache.mutable_data_ptr(), code_of(t), slots.const_data_ptr<int64_t>(), num_tokens,
                                  int(heads), int(d), int(block), num_blocks, key.stride(0), key.stride(1),
                                  value.stride(0), value.stride(1), k_cache.stride(0), k_cache.stride(1),
                                  k_cache.stride(2), v_cache.stride(0), v_cache.stride(1), v_cache.stride(2),
                                  stream_of(key)),
           "fxpr_reshape_and_cache");
}

}  // namespace

// (set while the library is loaded: whether the launchers below were registered)
static int launchers_registered = 0;
extern "C" int fxpr_torch_registered() { return launchers_registered; }

TORCH_LIBRARY_IMPL(fxpr, CUDA, m) {
  // another kernel library than the one compiled against: its entry points may
  // take other arguments. (No exception: none can pass the loader.)
  if (fxpr_abi_version() != FXPR_ABI_VERSION) return;
  launchers_registered = 1;
  m.impl("float_to_fixed", &float_to_fixed);
  m.impl("fixed_to_float", &fixed_to_float);
  m.impl("fixed_row_sum", &fixed_row_sum);
  m.impl("rms_norm_fxp", &rms_norm);
  m.impl("rms_norm_fxp_residual", &rms_norm_residual);
  m.impl("log_softmax_fxp", &log_softmax);
  m.impl("sample_greedy_fxp", &sample_greedy);
  m.impl("gemm_fxp", &gemm);
  m.impl("unified_attention_fxp", &unified_attention);
  m.impl("reshape_and_cache", &reshape_and_cache);
}
