// HPE with a lane per row: the kernels of many rows and short tables
// (hpe_rows.hip).
#ifndef MOPS_AMD_HPE_ROWS_HPP
#define MOPS_AMD_HPE_ROWS_HPP

#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "hpe_tiles.hpp"

namespace mops::amd::hpe_rows {

using hpe_tiles::Shape;

/// Whether the kernels hold the shape (the values of 64 rows fit in LDS).
bool covers_forward(const Shape& shape, size_t element_size);
bool covers_vjp(const Shape& shape, size_t element_size);

template <typename T>
void forward(T* output, const T* A, const T* C, const int32_t* P, const Shape& shape, hipStream_t stream);

/// `workspace`: hpe_tiles::table_bytes() bytes.
template <typename T>
void vjp(
    T* grad_A, const T* grad_output, const T* A, const T* C, const int32_t* P, const Shape& shape, void* workspace,
    hipStream_t stream
);

} // namespace mops::amd::hpe_rows

#endif
