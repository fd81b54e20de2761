// HPE with the values of a few rows in LDS and the monomials spread over a
// workgroup in teams of four lanes: the kernels of long tables (hpe_tiles.hip).
// hpe.hip calls them when `plan_*` finds a layout (orders 1 to 6, tiles that fit
// in LDS) and they are ahead of the others (thresholds::hpe_*).
#ifndef MOPS_AMD_HPE_TILES_HPP
#define MOPS_AMD_HPE_TILES_HPP

#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

namespace mops::amd::hpe_tiles {

struct Shape {
    int32_t n_rows;
    int32_t nA;
    int32_t n_monomials;
    int32_t order;
};

/// How a launch is cut: 4 * values rows per workgroup, `groups` workgroups per
/// tile of rows (shares of the monomials in the forward pass, of the features
/// in the gradients). values = 0: these kernels do not cover the shape.
struct Plan {
    int values = 0;
    int32_t tiles = 0;
    int32_t groups = 0;
    int log2_parts = 0; // teams that share the list of a feature
    size_t lds = 0;
};

/// Whether the kernels here and in hpe_rows.hip cover the table (orders 1 to 6, something to do).
bool covered(const Shape& shape);

/// Features up to which the table can be turned round (counters of the sort in LDS).
constexpr int32_t MAX_FEATURES = 10000;

/// The table turned round: for every feature the terms of its gradient. The
/// records of feature f are those from 4 lists[f] up to 4 lists[f + 1], each
/// the byte offsets of the order - 1 other factors (feature * stride; a factor
/// out of range counts as feature nA) and the coefficient behind them; lists
/// are filled up to four records with terms that are zero. For covered()
/// shapes of at most MAX_FEATURES features.
struct TurnedTable {
    int32_t* lists;
    int32_t* counts; // of the sort
    uint32_t* records;
};
size_t table_bytes(const Shape& shape, size_t element_size);
template <typename T>
TurnedTable turn_table(
    const T* C, const int32_t* P, const Shape& shape, int32_t stride, void* workspace, hipStream_t stream
);

Plan plan_forward(const Shape& shape, size_t element_size);
/// `second`: the second-order pass, which keeps two values per row and feature.
Plan plan_gradient(const Shape& shape, size_t element_size, bool second);

/// Scratch memory of a call (0 is possible for the forward pass).
size_t forward_bytes(const Shape& shape, const Plan& plan, size_t element_size);
size_t gradient_bytes(const Shape& shape, const Plan& plan, size_t element_size, bool second);

/// `counters`: at least plan.tiles zeros; they are zeros again at the end.
template <typename T>
void forward(
    T* output, const T* A, const T* C, const int32_t* P, const Shape& shape, const Plan& plan, void* workspace,
    int32_t* counters, hipStream_t stream
);

template <typename T>
void vjp(
    T* grad_A, const T* grad_output, const T* A, const T* C, const int32_t* P, const Shape& shape, const Plan& plan,
    void* workspace, hipStream_t stream
);

/// Either output may be null.
template <typename T>
void vjp_vjp(
    T* grad_grad_output, T* grad_A_2, const T* grad_grad_A, const T* grad_output, const T* A, const T* C,
    const int32_t* P, const Shape& shape, const Plan& plan, void* workspace, int32_t* counters, hipStream_t stream
);

} // namespace mops::amd::hpe_tiles

#endif
