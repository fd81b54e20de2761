// sap_rows.hpp for float.
#include "sap_rows_kernels.hpp"

namespace mops::amd::sap_rows {

template void forward<float>(
    float*, const float*, const float*, const float*, const float*, const Table&, const Shape&, hipStream_t
);
template void vjp<float>(
    float*, float*, const float*, const float*, const float*, const Table&, const Shape&, hipStream_t
);

} // namespace mops::amd::sap_rows
