// sap_rows.hpp for double.
#include "sap_rows_kernels.hpp"

namespace mops::amd::sap_rows {

template void forward<double>(
    double*, const double*, const double*, const double*, const double*, const Table&, const Shape&, hipStream_t
);
template void vjp<double>(
    double*, double*, const double*, const double*, const double*, const Table&, const Shape&, hipStream_t
);

} // namespace mops::amd::sap_rows
