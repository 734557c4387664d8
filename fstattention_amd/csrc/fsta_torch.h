// Host functions of the torch binding, shared by its operator registration and its Python module.
#pragma once

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>

#include <tuple>

namespace fsta_torch {

// An uninitialised tensor of the device's allocator, without the dispatcher's 0.4 us (every output here is written whole)
inline at::Tensor fresh(at::IntArrayRef sizes, at::ScalarType dtype, const at::Tensor& like) {
    return at::Tensor(at::detail::empty_cuda(sizes, dtype, like.device(), c10::nullopt));
}

// FSTA_* code of a storage type, -1 for types the library does not take
int dtype_code(at::ScalarType t);

// (o, lse or undefined); the checks raise ValueError
std::tuple<at::Tensor, at::Tensor> attention_fwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                                 const at::Tensor& ancestor_idx, const at::Tensor& mask_bits,
                                                 const at::Tensor& anc_count, const at::Tensor& leaf_idx,
                                                 const c10::optional<at::Tensor>& plan, int64_t key_shift,
                                                 double sm_scale, int64_t block_m, int64_t max_ancestors,
                                                 int64_t out_dtype_code, bool return_lse, int64_t flags,
                                                 const c10::optional<at::Tensor>& k_scale,
                                                 const c10::optional<at::Tensor>& v_scale);

}  // namespace fsta_torch
