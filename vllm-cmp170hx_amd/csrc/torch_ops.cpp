// The operators a decode step calls, in host-only C++ (g++, no device code):
//  * the CUDA-key implementations of _exl3_C's linear_out and moe_out family: the
//    tensor checks of csrc/exl3/common.h:42-61, dense.cu:85-93 and
//    moe.cu:323-364 with the reference's messages, then the C-ABI entry point on
//    torch's current stream (schemas: vllm_mi355x/kernels/exl3/_C.py);
//  * _vllm_mi355x::marlin_moe, the launches of one fused Marlin MoE call on the
//    path and buffers that kernels/marlin_moe/fused.py chose.
// From Python the same checks and calls took longer than the kernels of a small
// call: a 5120 x 512 linear of one row 21.6 us a call (6 on the GPU), 10.2
// with its operator here; the fused MoE of 48 tokens 85 us of host work for four
// or five launches.
//
// The loader (vllm_mi355x/_native.py) names the loaded libvllm_mi355x.so
// (vllm_mi355x_torch_bind), so that operators and ctypes calls always run in one
// library.
#include <ATen/core/Tensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/library.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <initializer_list>
#include <optional>

#include "../../include/vllm_mi355x.h"

namespace {

decltype(&exl3_linear_out) native_linear_out = nullptr;
decltype(&exl3_moe_out) native_moe_out = nullptr;
decltype(&moe_align_block_size) native_align = nullptr;
decltype(&marlin_moe_align_permute) native_align_permute = nullptr;
decltype(&marlin_moe_gemm) native_gemm = nullptr;
decltype(&marlin_moe_gemm_direct) native_gemm_direct = nullptr;
decltype(&marlin_moe_w13_act) native_w13_act = nullptr;
decltype(&marlin_moe_w2_sum) native_w2_sum = nullptr;
decltype(&marlin_moe_rows) native_rows = nullptr;
decltype(&moe_sum) native_sum = nullptr;
decltype(&vllm_mi355x_last_error) native_last_error = nullptr;

int dtype_code(at::ScalarType t) {
  return t == at::kBFloat16 ? VQ_BF16 : (t == at::kHalf ? VQ_FP16 : VQ_FP32);
}

void check_tensor(const at::Tensor& t, const at::Tensor& x, std::initializer_list<at::ScalarType> dtypes,
                  const char* name) {
  TORCH_CHECK(t.is_cuda() && t.device() == x.device(), name, " must be on the input CUDA device");
  bool known = false;
  for (at::ScalarType d : dtypes) known = known || t.scalar_type() == d;
  TORCH_CHECK(known, name, " has incorrect dtype");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

void check_integer(const at::Tensor& t, const at::Tensor& x, const char* name) {
  TORCH_CHECK(t.scalar_type() == at::kInt || t.scalar_type() == at::kLong, name, " must have int32 or int64 dtype");
  check_tensor(t, x, {t.scalar_type()}, name);
}

void* stream_of(const at::Tensor& x) { return c10::hip::getCurrentHIPStream(x.device().index()).stream(); }

void check_status(int status) { TORCH_CHECK(status == 0, native_last_error()); }

void linear_out(const at::Tensor& x, const at::Tensor& trellis, const at::Tensor& suh, const at::Tensor& svh,
                int64_t bits_x2, int64_t codebook, int64_t logical_in, int64_t logical_out,
                const at::Tensor& out, const at::Tensor& workspace) {
  TORCH_CHECK(x.is_cuda(), "EXL3 x must be CUDA");
  check_tensor(x, x, {at::kBFloat16, at::kHalf}, "x");
  check_tensor(trellis, x, {at::kShort}, "trellis");
  check_tensor(suh, x, {at::kHalf}, "suh");
  check_tensor(svh, x, {at::kHalf}, "svh");
  TORCH_CHECK(out.scalar_type() == at::kBFloat16 || out.scalar_type() == at::kHalf || out.scalar_type() == at::kFloat,
              "EXL3 linear out must be BF16, FP16 or FP32");
  check_tensor(out, x, {out.scalar_type()}, "out");
  check_tensor(workspace, x, {at::kFloat}, "workspace");
  TORCH_CHECK(x.dim() == 2 && trellis.dim() == 3 && suh.dim() == 1 && svh.dim() == 1 && out.dim() == 2,
              "EXL3 linear requires rank-2 x/out, rank-3 trellis and rank-1 scales");
  const c10::DeviceGuard guard(x.device());
  check_status(native_linear_out(
      x.const_data_ptr(), dtype_code(x.scalar_type()), x.size(0), x.size(1), trellis.const_data_ptr(), trellis.size(0),
      trellis.size(1), trellis.size(2), suh.const_data_ptr(), suh.numel(), svh.const_data_ptr(), svh.numel(), bits_x2,
      codebook, logical_in, logical_out, out.mutable_data_ptr(), dtype_code(out.scalar_type()), out.size(0),
      out.size(1), static_cast<float*>(workspace.mutable_data_ptr()), workspace.numel(), stream_of(x)));
}

void moe(const at::Tensor& x, const at::Tensor& topk_ids, const at::Tensor& topk_weights,
         const at::Tensor& packed_ptrs, const at::Tensor& packed_meta, const at::Tensor& expert_map,
         int64_t intermediate_size, int64_t bits_x2, const at::Tensor& out, const at::Tensor& workspace,
         double swiglu_limit) {
  TORCH_CHECK(x.is_cuda(), "EXL3 x must be CUDA");
  check_tensor(x, x, {at::kBFloat16, at::kHalf}, "x");
  check_integer(topk_ids, x, "topk_ids");
  check_integer(expert_map, x, "expert_map");
  check_tensor(topk_weights, x, {at::kFloat}, "topk_weights");
  check_tensor(packed_ptrs, x, {at::kLong}, "packed_ptrs");
  check_tensor(packed_meta, x, {at::kLong}, "packed_meta");
  check_tensor(out, x, {x.scalar_type()}, "out");
  check_tensor(workspace, x, {at::kFloat}, "workspace");
  TORCH_CHECK(x.dim() == 2 && out.dim() == 2 && topk_ids.dim() == 2 && topk_weights.dim() == 2 &&
                  expert_map.dim() == 1 && packed_ptrs.dim() == 3 && packed_meta.dim() == 3,
              "EXL3 MoE tensor ranks mismatch");
  const int64_t rows = x.size(0), experts = packed_ptrs.size(0);
  TORCH_CHECK(topk_ids.size(0) == rows && topk_weights.sizes() == topk_ids.sizes() && out.sizes() == x.sizes(),
              "EXL3 MoE row/topk/output geometry mismatch");
  TORCH_CHECK(packed_ptrs.size(1) == 3 && packed_ptrs.size(2) == 3 && packed_meta.size(0) == experts &&
                  packed_meta.size(1) == 3 && packed_meta.size(2) == 4,
              "EXL3 MoE pointer/metadata geometry mismatch");
  const c10::DeviceGuard guard(x.device());
  check_status(native_moe_out(
      x.const_data_ptr(), dtype_code(x.scalar_type()), rows, x.size(1), topk_ids.const_data_ptr(),
      topk_ids.scalar_type() == at::kLong, static_cast<const float*>(topk_weights.const_data_ptr()), topk_ids.size(1),
      static_cast<const int64_t*>(packed_ptrs.const_data_ptr()),
      static_cast<const int64_t*>(packed_meta.const_data_ptr()), experts, expert_map.const_data_ptr(),
      expert_map.scalar_type() == at::kLong, expert_map.numel(), intermediate_size, bits_x2, out.mutable_data_ptr(),
      dtype_code(out.scalar_type()), static_cast<float*>(workspace.mutable_data_ptr()), workspace.numel(),
      static_cast<float>(swiglu_limit), stream_of(x)));
}

// moe_out: each matrix's own format.
void moe_out(const at::Tensor& x, const at::Tensor& topk_ids, const at::Tensor& topk_weights,
             const at::Tensor& packed_ptrs, const at::Tensor& packed_meta, const at::Tensor& expert_map,
             int64_t intermediate_size, const at::Tensor& out, const at::Tensor& workspace, double swiglu_limit) {
  moe(x, topk_ids, topk_weights, packed_ptrs, packed_meta, expert_map, intermediate_size, 0, out, workspace,
      swiglu_limit);
}

// moe_out's schema at the one rate the reference's prefill operator is built
// for (csrc/exl3/moe_prefill.cu:37-40, :169-171).
void moe_out_prefill(const at::Tensor& x, const at::Tensor& topk_ids, const at::Tensor& topk_weights,
                     const at::Tensor& packed_ptrs, const at::Tensor& packed_meta, const at::Tensor& expert_map,
                     int64_t intermediate_size, const at::Tensor& out, const at::Tensor& workspace,
                     double swiglu_limit) {
  constexpr int64_t kPrefillBitsX2 = 10;
  moe(x, topk_ids, topk_weights, packed_ptrs, packed_meta, expert_map, intermediate_size, kPrefillBitsX2, out,
      workspace, swiglu_limit);
}

// moe_out_v2: one mul1 rate for the layer.
void moe_out_v2(const at::Tensor& x, const at::Tensor& topk_ids, const at::Tensor& topk_weights,
                const at::Tensor& packed_ptrs, const at::Tensor& packed_meta, const at::Tensor& expert_map,
                int64_t intermediate_size, int64_t bits_x2, const at::Tensor& out, const at::Tensor& workspace,
                double swiglu_limit) {
  TORCH_CHECK(bits_x2 > 0, "EXL3 MoE v2 needs the layer's bits_x2");
  moe(x, topk_ids, topk_weights, packed_ptrs, packed_meta, expert_map, intermediate_size, bits_x2, out, workspace,
      swiglu_limit);
}

// The _mixed variants: every expert's own format, whatever rate is named.
void moe_out_v2_mixed(const at::Tensor& x, const at::Tensor& topk_ids, const at::Tensor& topk_weights,
                      const at::Tensor& packed_ptrs, const at::Tensor& packed_meta, const at::Tensor& expert_map,
                      int64_t intermediate_size, int64_t bits_x2, const at::Tensor& out, const at::Tensor& workspace,
                      double swiglu_limit) {
  (void)bits_x2;
  moe(x, topk_ids, topk_weights, packed_ptrs, packed_meta, expert_map, intermediate_size, 0, out, workspace,
      swiglu_limit);
}

// One fused Marlin MoE call (kernels/marlin_moe/fused.py): path 0 staged (block
// alignment, w13 partials with their SwiGLU, w2), 1 direct (alignment and
// k-permuted activations, w13 with the SwiGLU, w2), 2 row lists, 3 one token's
// identity routing (w13 partials with their SwiGLU, w2 with the slot sum); then,
// but for 3, the slot-order sum.  ids: int32 local experts [M, topk].  lists:
// the aligned slots (row lists: the table); act: FP32 w13 partials (0, 3) or the
// k-permuted activations (1, 2).
void marlin_moe(const at::Tensor& x, const at::Tensor& w1, const at::Tensor& w2, const at::Tensor& s1,
                const at::Tensor& s2, const at::Tensor& topk_w, const at::Tensor& ids, int64_t path,
                int64_t block_size, int64_t ksplit, double limit, const std::optional<at::Tensor>& lists,
                const std::optional<at::Tensor>& expert_ids, const std::optional<at::Tensor>& ntpp,
                const at::Tensor& act, const at::Tensor& h, const at::Tensor& c3, const at::Tensor& out) {
  const int64_t m = x.size(0), k = x.size(1), experts = w1.size(0), n = w2.size(1) * 16, topk = ids.size(1);
  const int64_t slots = m * topk;
  const at::ScalarType type = x.scalar_type();
  TORCH_CHECK((type == at::kBFloat16 || type == at::kHalf) && x.dim() == 2 && x.stride(1) == 1,
              "a: bf16 or fp16, unit inner stride");
  TORCH_CHECK(s1.scalar_type() == type && s2.scalar_type() == type, "scales must have the activation dtype");
  TORCH_CHECK(w1.scalar_type() == at::kInt && w1.is_contiguous() && s1.is_contiguous() &&
                  w2.scalar_type() == at::kInt && w2.is_contiguous() && s2.is_contiguous(),
              "weights contiguous");
  TORCH_CHECK(w1.dim() == 3 && w1.size(1) * 16 == k && w1.size(2) == 4 * n && w2.dim() == 3 && w2.size(0) == experts &&
                  w2.size(2) == 2 * k,
              "w: int32 [E, K/16, 2N]");
  TORCH_CHECK(s1.dim() == 3 && s1.size(0) == experts && s1.size(1) * 128 == k && s1.size(2) == 2 * n && s2.dim() == 3 &&
                  s2.size(0) == experts && s2.size(1) * 128 == n && s2.size(2) == k,
              "s: [E, K/128, N]");
  TORCH_CHECK(ids.scalar_type() == at::kInt && ids.is_contiguous() && ids.numel() == slots, "routing dtypes");
  TORCH_CHECK(topk_w.scalar_type() == at::kFloat && topk_w.is_contiguous() && topk_w.numel() == slots,
              "topk weights fp32");
  TORCH_CHECK(out.scalar_type() == type && out.is_contiguous() &&
                  (path == 3 ? out.numel() >= k : out.sizes() == x.sizes()),
              "moe_sum: out must be a contiguous [M, H] of the input dtype");
  for (const at::Tensor* t : {&w1, &w2, &s1, &s2, &topk_w, &ids, &act, &h, &c3, &out}) {
    TORCH_CHECK(t->is_cuda() && t->device() == x.device(), "tensors must be on the activation device");
  }
  TORCH_CHECK(h.scalar_type() == type && h.is_contiguous() && h.numel() >= slots * n, "act: buffers too small");
  TORCH_CHECK(c3.scalar_type() == type && c3.is_contiguous() && c3.numel() >= slots * k, "output too small");
  const bool permuted = path == 1 || path == 2;
  TORCH_CHECK(act.is_contiguous() && act.scalar_type() == (permuted ? type : at::kFloat), "w13 partial buffer");
  TORCH_CHECK(!permuted || act.numel() >= m * k, "permute: output too small");
  for (const std::optional<at::Tensor>* t : {&lists, &expert_ids, &ntpp}) {
    TORCH_CHECK(!t->has_value() || ((*t)->scalar_type() == at::kInt && (*t)->is_contiguous() && (*t)->is_cuda() &&
                                    (*t)->device() == x.device()),
                "routing dtypes");
  }
  const c10::DeviceGuard guard(x.device());
  void* stream = stream_of(x);
  const int dtype = dtype_code(type);
  const auto words = [](const at::Tensor& t) { return static_cast<const int32_t*>(t.const_data_ptr()); };
  const int32_t* routed = words(ids);
  const float* weights = static_cast<const float*>(topk_w.const_data_ptr());
  if (path == 2) {
    TORCH_CHECK(lists.has_value(), "routing dtypes");
    check_status(native_rows(x.const_data_ptr(), dtype, m, x.stride(0), words(w1), s1.const_data_ptr(), words(w2),
                             s2.const_data_ptr(), experts, routed, weights, topk, k, n, static_cast<float>(limit),
                             block_size, static_cast<int32_t*>(lists->mutable_data_ptr()), lists->numel(),
                             act.mutable_data_ptr(), h.mutable_data_ptr(), c3.mutable_data_ptr(), stream));
  } else {
    int32_t* sorted = nullptr;
    int32_t* eids = nullptr;
    int32_t* padded = nullptr;
    int64_t sorted_numel = 0, blocks = 0;
    if (path != 3) {
      // upstream moe_align_block_size's output sizes
      sorted_numel = slots + experts * (block_size - 1);
      if (slots < experts) sorted_numel = std::min(slots * block_size, sorted_numel);
      blocks = (sorted_numel + block_size - 1) / block_size;
      TORCH_CHECK(lists.has_value() && expert_ids.has_value() && ntpp.has_value() && lists->numel() >= sorted_numel &&
                      expert_ids->numel() >= blocks && ntpp->numel() >= 1,
                  "align: buffers too small");
      sorted = static_cast<int32_t*>(lists->mutable_data_ptr());
      eids = static_cast<int32_t*>(expert_ids->mutable_data_ptr());
      padded = static_cast<int32_t*>(ntpp->mutable_data_ptr());
    }
    if (path == 1) {
      check_status(native_align_permute(routed, slots, experts, block_size, nullptr, sorted, sorted_numel, eids, blocks,
                                        padded, x.const_data_ptr(), dtype, m, k, x.stride(0), act.mutable_data_ptr(), k,
                                        stream));
      constexpr int kSwiglu = 3;
      check_status(native_gemm_direct(act.const_data_ptr(), dtype, m, k, words(w1), s1.const_data_ptr(), experts, sorted,
                                      sorted_numel, eids, blocks, padded, nullptr, topk, slots, k, 2 * n, block_size,
                                      kSwiglu, 1, static_cast<float>(limit), nullptr, 0, h.mutable_data_ptr(), n, slots,
                                      stream));
    } else {
      float* part = static_cast<float*>(act.mutable_data_ptr());
      const int32_t* owners = routed;  // identity routing: slot b is block b
      int64_t owner_numel = slots;
      if (path == 0) {
        check_status(native_align(routed, slots, experts, block_size, nullptr, sorted, sorted_numel, eids, blocks, padded,
                                  stream));
        owners = eids;
        owner_numel = blocks;
      }
      check_status(native_w13_act(x.const_data_ptr(), dtype, m, x.stride(0), words(w1), s1.const_data_ptr(), experts,
                                  sorted, sorted_numel, owners, owner_numel, padded, routed, topk, slots, k, 2 * n,
                                  block_size, ksplit, static_cast<float>(limit), part, act.numel(),
                                  h.mutable_data_ptr(), n, slots, stream));
      if (path == 3) {
        check_status(native_w2_sum(h.const_data_ptr(), dtype, slots, n, words(w2), s2.const_data_ptr(), experts, routed,
                                   slots, weights, topk, slots, n, k, block_size, c3.mutable_data_ptr(), k, slots,
                                   out.mutable_data_ptr(), stream));
        return;
      }
    }
    constexpr int kTopk = 2;
    if (path == 1) {
      check_status(native_gemm_direct(h.const_data_ptr(), dtype, slots, n, words(w2), s2.const_data_ptr(), experts, sorted,
                                      sorted_numel, eids, blocks, padded, weights, 1, slots, n, k, block_size, kTopk, 1,
                                      INFINITY, nullptr, 0, c3.mutable_data_ptr(), k, slots, stream));
    } else {
      check_status(native_gemm(h.const_data_ptr(), dtype, slots, n, words(w2), s2.const_data_ptr(), experts, sorted,
                               sorted_numel, eids, blocks, padded, weights, 1, slots, n, k, block_size, kTopk, 1, nullptr,
                               0, c3.mutable_data_ptr(), k, slots, stream));
    }
  }
  check_status(native_sum(c3.const_data_ptr(), dtype, m, topk, k, routed, experts, out.mutable_data_ptr(), stream));
}

template <typename F>
bool find(void* library, const char* name, F& f) {
  f = reinterpret_cast<F>(dlsym(library, name));
  return f != nullptr;
}

}  // namespace

// The entry points of the loaded library (its dlopen handle); 0, or 1 when one
// is missing.
extern "C" int vllm_mi355x_torch_bind(void* library) {
  const bool all = find(library, "exl3_linear_out", native_linear_out) && find(library, "exl3_moe_out", native_moe_out) &&
                   find(library, "moe_align_block_size", native_align) &&
                   find(library, "marlin_moe_align_permute", native_align_permute) &&
                   find(library, "marlin_moe_gemm", native_gemm) &&
                   find(library, "marlin_moe_gemm_direct", native_gemm_direct) &&
                   find(library, "marlin_moe_w13_act", native_w13_act) &&
                   find(library, "marlin_moe_w2_sum", native_w2_sum) && find(library, "marlin_moe_rows", native_rows) &&
                   find(library, "moe_sum", native_sum) && find(library, "vllm_mi355x_last_error", native_last_error);
  return all ? 0 : 1;
}

TORCH_LIBRARY_IMPL(_exl3_C, CUDA, m) {
  m.impl("linear_out", &linear_out);
  m.impl("linear_out_splitk", &linear_out);
  m.impl("linear_out_prefill", &linear_out);
  m.impl("moe_out", &moe_out);
  m.impl("moe_out_mixed", &moe_out);
  m.impl("moe_out_prefill", &moe_out_prefill);
  m.impl("moe_out_v2", &moe_out_v2);
  m.impl("moe_out_v2_fold", &moe_out_v2);
  m.impl("moe_out_prefill_v2", &moe_out_v2);
  m.impl("moe_out_prefill_try", &moe_out_v2);
  m.impl("moe_out_v2_try", &moe_out_v2);
  m.impl("moe_out_v2_try_mixed", &moe_out_v2);
  m.impl("moe_out_v2_mixed", &moe_out_v2_mixed);
  m.impl("moe_out_prefill_try_mixed", &moe_out_v2_mixed);
}

TORCH_LIBRARY(_vllm_mi355x, m) {
  m.def(
      "marlin_moe(Tensor x, Tensor w1, Tensor w2, Tensor s1, Tensor s2, Tensor topk_w, Tensor ids, int path, "
      "int block_size, int ksplit, float limit, Tensor(a!)? lists, Tensor(b!)? expert_ids, Tensor(c!)? ntpp, "
      "Tensor(d!) act, Tensor(e!) h, Tensor(f!) c3, Tensor(g!) out) -> ()");
}

TORCH_LIBRARY_IMPL(_vllm_mi355x, CUDA, m) { m.impl("marlin_moe", &marlin_moe); }
// an inference call: inputs that require gradients are read as they are
TORCH_LIBRARY_IMPL(_vllm_mi355x, Autograd, m) { m.impl("marlin_moe", torch::CppFunction::makeFallthrough()); }
