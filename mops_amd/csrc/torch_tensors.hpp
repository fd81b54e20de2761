// What the callers of this library on PyTorch tensors (torch_ops.cpp,
// array_ops.cpp) share: views, the stream, and outputs.
#ifndef MOPS_AMD_TORCH_TENSORS_HPP
#define MOPS_AMD_TORCH_TENSORS_HPP

#include <stdexcept>
#include <string>

#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/types.h>

#include "mops/amd.h"
#include "mops/tensor.hpp"

namespace mops::amd::torch_tensors {

template <typename T, size_t N> mops::Tensor<T, N> view(const at::Tensor& tensor, const char* name) {
    mops::Tensor<T, N> result{nullptr, {}};
    for (size_t d = 0; d < N; d++) {
        result.shape[d] = 0;
    }
    if (!tensor.defined()) {
        return result; // "not wanted" / "not given": a null view
    }
    if (static_cast<size_t>(tensor.dim()) != N) {
        throw std::runtime_error(
            std::string(name) + " must have " + std::to_string(N) + " dimensions, got " + std::to_string(tensor.dim())
        );
    }
    result.data = tensor.data_ptr<T>();
    for (size_t d = 0; d < N; d++) {
        result.shape[d] = static_cast<size_t>(tensor.size(static_cast<int64_t>(d)));
    }
    return result;
}

/// The library's launches go to PyTorch's current stream of the tensors' device, without blocking.
/// (In a ROCm build of PyTorch the HIP device type goes under the name of CUDA: these are the
/// guard and the stream of that build.)
struct OnTorchStream {
    c10::hip::HIPGuardMasqueradingAsCUDA guard;
    explicit OnTorchStream(const at::Tensor& tensor) : guard(tensor.device()) {
        mops_amd_set_stream(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream());
        mops_amd_set_synchronous(0);
    }
};

template <typename Body> void by_dtype(const at::Tensor& like, Body&& body) {
    if (like.scalar_type() == at::kFloat) {
        body(float{});
    } else {
        body(double{});
    }
}

/// An uninitialised tensor beside `like` (the library overwrites its outputs completely), from the
/// caching allocator without a turn through the dispatcher: 0.5 us instead of 0.7.
inline at::Tensor new_tensor(at::IntArrayRef sizes, const at::Tensor& like) {
    return at::detail::empty_cuda(
        sizes, like.scalar_type(), c10::nullopt, like.device(), c10::nullopt, c10::nullopt
    );
}
inline at::Tensor new_like(const at::Tensor& like) { return new_tensor(like.sizes(), like); }

} // namespace mops::amd::torch_tensors

#endif
