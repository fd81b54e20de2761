// SAP with a lane per row, for batches that fill the device that way
// (sap_rows.hip). sap.hip calls these when the rules below say so.
#ifndef MOPS_AMD_SAP_ROWS_HPP
#define MOPS_AMD_SAP_ROWS_HPP

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "dispatch_thresholds.hpp"
#include "sap_mfma.hpp"

namespace mops::amd::sap_rows {

using sap_mfma::Shape;
using sap_mfma::Table;

constexpr int32_t MAX_ENTRIES = 32 * 1024; // of the table
constexpr int32_t MOST_INNER = 16;         // values of the inner index: of the one that pads better
constexpr int32_t MOST_OUTER = 24;         // values of the other: in LDS, with their gradients

/// Columns of the result that a lane works on at a time (rows of M as long as two of them fit the scalar
/// registers), and how many such tiles there are.
struct Tiles {
    int32_t columns, count;
};
inline Tiles tiles_of(int32_t n_out, size_t element_size) {
    const int32_t most = element_size == 4 ? 32 : 20;
    const int32_t count = (n_out + most - 1) / most;
    return Tiles{((n_out + count - 1) / count + 3) / 4 * 4, count};
}
inline int32_t padded(int32_t n_inner) { return std::max(4, (n_inner + 1) / 2 * 2); }

/// Whether A's index is the inner one: the one whose padding costs less, and fits.
inline bool inner_is_A(const Shape& s) {
    if (s.nA > MOST_INNER || s.nB > MOST_INNER) {
        return s.nA <= MOST_INNER;
    }
    return padded(s.nA) * s.nB < padded(s.nB) * s.nA;
}

/// Elements of M as these kernels hold it.
inline int64_t cells(const Shape& s) {
    const Tiles tiles = tiles_of(s.nO, sizeof(double));
    return static_cast<int64_t>(inner_is_A(s) ? padded(s.nA) * s.nB : padded(s.nB) * s.nA) * tiles.columns * tiles.count;
}
inline bool covers(const Shape& s) {
    return s.n_rows >= 1 && s.nA >= 1 && s.nB >= 1 && s.nO >= 1 && std::min(s.nA, s.nB) <= MOST_INNER &&
           std::max(s.nA, s.nB) <= MOST_OUTER && s.K >= 1 && s.K <= MAX_ENTRIES;
}

/// The rules. What a lane per row costs: 4 cycles per cell of M for 64 rows; the matrix cores, 128 (double
/// 256) per step of 4 x 16 x 16; the table in global memory and a lane per row and column, as many LDS
/// reads as there are entries.
inline bool chosen_vjp(const Shape& s, size_t element_size) {
    if (!covers(s)) {
        return false;
    }
    if (!sap_mfma::supports_vjp(s, element_size)) {
        return s.n_rows >= thresholds::SAP_ROWS_BEYOND_MATRIX_CORES_VJP && cells(s) <= 10 * static_cast<int64_t>(s.K);
    }
    const bool cached = cells(s) * static_cast<int64_t>(element_size) <= thresholds::SAP_ROWS_CACHED_TABLE;
    const int64_t by_matrix = static_cast<int64_t>(s.nA + s.nB) * ((s.nO + 3) / 4) * (element_size == 4 ? 128 : 256);
    return s.n_rows >= (element_size == 8 && cached ? thresholds::SAP_ROWS_VJP / 2 : thresholds::SAP_ROWS_VJP) &&
           4 * cells(s) <= 0.8 * by_matrix;
}
inline bool chosen_forward(const Shape& s, size_t element_size) {
    if (!covers(s)) {
        return false;
    }
    if (!sap_mfma::supports_forward(s, element_size)) {
        return s.n_rows >= thresholds::SAP_ROWS_BEYOND_MATRIX_CORES && cells(s) <= 6 * static_cast<int64_t>(s.K);
    }
    const bool cached = cells(s) * static_cast<int64_t>(element_size) <= thresholds::SAP_ROWS_CACHED_TABLE;
    const int64_t by_matrix =
        static_cast<int64_t>(s.nA) * ((s.nB + 3) / 4) * ((s.nO + 15) / 16) * (element_size == 4 ? 128 : 256);
    return s.n_rows >= thresholds::SAP_ROWS_FORWARD && cached && 4 * cells(s) <= 0.6 * by_matrix;
}
/// Of the forward pass of two pairs, which the matrix cores have in one launch only for smaller batches.
inline bool chosen_forward_of_two_pairs(const Shape& s, size_t element_size) {
    return chosen_forward(s, element_size) ||
           (covers(s) && sap_mfma::supports_forward(s, element_size) && s.n_rows >= thresholds::SAP_ROWS_VJP);
}

/// Scratch memory of a call: M, and a row that is only asked for.
inline size_t scratch_bytes(const Shape& s, size_t element_size) {
    const Tiles tiles = tiles_of(s.nO, element_size);
    const bool A_inside = inner_is_A(s);
    const size_t cells = static_cast<size_t>(padded(A_inside ? s.nA : s.nB)) * tiles.columns;
    return (static_cast<size_t>(tiles.count) * (A_inside ? s.nB : s.nA) * cells + tiles.columns) * element_size;
}

/// output = sap(A, B), or sap(A, B) + sap(A2, B2) when A2 is not null.
template <typename T>
void forward(
    T* output, const T* A, const T* B, const T* A2, const T* B2, const Table& table, const Shape& shape,
    hipStream_t stream
);

/// grad_A or grad_B may be null.
template <typename T>
void vjp(
    T* grad_A, T* grad_B, const T* grad_output, const T* A, const T* B, const Table& table, const Shape& shape,
    hipStream_t stream
);

} // namespace mops::amd::sap_rows

#endif
