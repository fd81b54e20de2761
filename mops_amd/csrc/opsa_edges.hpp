// The gradients of OPSA / OPSAW that belong to an edge each (opsa_edges.hip).
#ifndef MOPS_AMD_OPSA_EDGES_HPP
#define MOPS_AMD_OPSA_EDGES_HPP

#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "sender_shares.hpp"

namespace mops::amd::opsa_edges {

template <typename T> struct Tensors {
    T* grad_A; // [n_edges][K], may be null
    T* grad_B; // [n_edges][L], may be null
    T* edge_W; // [n_edges][L] what the edge adds to grad_W, may be null
    const T* grad_output; // [n_nodes][K][L]
    const T* A;
    const T* B;
    const T* W;               // [n_nodes][L]; null: OPSA
    const int32_t* receivers; // [n_edges], equal ones next to each other
    const int32_t* senders;   // [n_edges] (with W)
    int32_t n_edges, n_nodes, K, L;
};

/// Up to 32 columns of A and 64 of B.
bool covers(int32_t n_nodes, int32_t K, int32_t L, size_t element_size);

/// With `slots` and `slot_counts`, the edges of every sender are listed as well: by `list_blocks`
/// workgroups (sender_slots_blocks()) beside the others, or, if that is 0, by arrival
/// (SenderArrivals, one copy of the counters). With `plan` (or null), the senders are split into `shares`.
template <typename T>
void launch(
    const Tensors<T>& tensors, int32_t* slots, int32_t* slot_counts, unsigned list_blocks, const SharePlan* plan,
    const Shares& shares, hipStream_t stream
);

} // namespace mops::amd::opsa_edges

#endif
