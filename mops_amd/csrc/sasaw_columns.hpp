// SASAW with a lane per feature column (sasaw_columns.hip): the numbers of
// components of equivariant message passing. sasaw_segments.hip calls these for
// them and keeps its own kernels for other numbers.
#ifndef MOPS_AMD_SASAW_COLUMNS_HPP
#define MOPS_AMD_SASAW_COLUMNS_HPP

#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "dispatch_thresholds.hpp"
#include "sasaw_mfma.hpp"
#include "sender_buckets.hpp"
#include "sender_shares.hpp"

namespace mops::amd::sasaw_columns {

using sasaw_mfma::Indices;
using sasaw_mfma::Shape;

/// Whether these kernels cover sums over `nA` components and `block_rows` block
/// rows with `result_rows` rows of the result: 4, 9 or 16 of the first two (the
/// components of spherical harmonics up to some degree), at most 16 of the last.
bool covers(int32_t nA, int32_t block_rows, int32_t result_rows);

/// Where the matrix cores (sasaw_segments.hip) stay ahead in the forward pass:
/// 16 components in float leave none of their rows unused, and up to 16 columns
/// leave these kernels their narrowest tiles.
inline bool slower_forward(const Shape& shape, size_t element_size) {
    return element_size == 4 && shape.nA == 16 && shape.L <= 16 && shape.n_edges > thresholds::COLUMNS_EDGES_AT_16;
}

template <typename T>
void forward(
    T* output, const T* A, const T* B, const T* C, const T* W, const Indices& indices, const Shape& shape,
    hipStream_t stream
);

/// How the edges of every sender are found for grad_W: in shares and buckets (sender_shares.hpp) which
/// the launch for grad_A and grad_B splits the index into, or, if not in_shares, by a counting sort.
struct SenderLists {
    SharePlan plan;
    int32_t copies; // workgroups with the same bucket
    bool in_shares;
    size_t bytes() const { return shares_bytes(plan, copies); }
};
template <typename T> SenderLists plan_lists(const Shape& shape);

/// grad_A, grad_B: either may be null, but not both. `lists`: those to begin in `workspace`, or null.
template <typename T>
void edge_gradients(
    T* grad_A, T* grad_B, const T* grad_output, const T* A, const T* B, const T* C, const T* W, const Indices& indices,
    const Shape& shape, const SenderLists* lists, void* workspace, hipStream_t stream
);

/// The edges of every sender in the lists begun in `workspace`, or in the order of their senders: one of the
/// two is null.
template <typename T>
void weight_gradient(
    T* grad_W, const T* grad_output, const T* A, const T* B, const T* C, const Indices& indices, const Shape& shape,
    const SenderLists* lists, void* workspace, const EdgesBySender* ordered, hipStream_t stream
);

/// Whether a graph is small enough that all its gradients are one launch, in which every sender's edges are
/// looked for in the index as it is. Whichever of the gradients are wanted, so that the bits
/// of one do not depend on the others.
bool small(const Shape& shape, size_t element_size);

/// Of a small graph: any of grad_A, grad_B, grad_W may be null, but not all.
template <typename T>
void small_vjp(
    T* grad_A, T* grad_B, T* grad_W, const T* grad_output, const T* A, const T* B, const T* C, const T* W,
    const Indices& indices, const Shape& shape, hipStream_t stream
);

} // namespace mops::amd::sasaw_columns

#endif
