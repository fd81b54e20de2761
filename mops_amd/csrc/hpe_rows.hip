// Homogeneous polynomial evaluation with many rows and a short table, for
// gfx950 (semantics: hpe.hip).
//
// A lane is a row (or two: lane and lane + 64, where the tile of 128 rows fits
// in LDS) and all lanes of a wavefront are at the same monomial: a batch of 64
// table entries is loaded one per lane and handed out through readlane. The
// tile of A is feature by feature, the rows side by side, with one feature
// more, all zero, that stands for a factor outside the tensor. One fixed order
// of summation, no atomics.
//
// Against hpe_tiles.hip, whose workgroup has 16 rows or fewer and 256 teams for
// the monomials, most of which a short table leaves idle. What bounds these
// kernels is LDS (a value per row and factor) and the readlanes that hand the
// entries out, for wide rows the filling of the tile. 100 000 rows, whole calls,
// hpe_tiles.hip / this file, us: 10 features, 50 monomials of order 3, forward
// 27.5 / 8.0 (float), 41.6 / 11.4 (double), vjp 42.5 / 15.2 and 87 / 17.7; 100
// features, 300 of order 2, forward 40.2 / 19.8 and 66 / 32. Which of them a call
// takes: thresholds::hpe_forward and hpe_vjp (dispatch_thresholds.hpp).
#include <algorithm>
#include <type_traits>

#include "hpe_rows.hpp"

#include "device_common.hpp"
#include "runtime.hpp"

namespace mops::amd {
namespace hpe_rows {
namespace {

constexpr int WAVES = 16;
constexpr int THREADS = WAVES * WAVE;
constexpr size_t LDS_LIMIT = 140 * 1024; // of the 160 KB of a compute unit

/// Rows per workgroup when a lane has RPL of them: the table entry a wavefront is at then serves
/// RPL rows per lane for the same readlanes and address.
__host__ __device__ constexpr int rows_of(int rpl) { return WAVE * rpl; }
/// Distance between features in the tile of A (odd: the values of a row are stored on different banks).
__host__ __device__ constexpr int pitch_of(int rpl) { return WAVE * rpl + 1; }

/// The values of the workgroup's rows, feature by feature, and the zeros of feature nA.
template <typename T, int RPL>
__device__ __forceinline__ void stage(T* tile, const T* __restrict__ A, int32_t row0, int32_t rows, int32_t nA) {
    constexpr int ROWS = rows_of(RPL), PITCH = pitch_of(RPL), LOADS = 4;
    const int tid = threadIdx.x;
    const T* from = A + static_cast<size_t>(row0) * nA;
    for (int32_t i0 = tid; i0 < ROWS * nA; i0 += LOADS * THREADS) {
        T value[LOADS];
#pragma unroll
        for (int u = 0; u < LOADS; u++) {
            const int32_t i = i0 + u * THREADS;
            value[u] = load_or_zero(from, static_cast<size_t>(i), i < rows * nA); // rows beyond the end: zeros
        }
#pragma unroll
        for (int u = 0; u < LOADS; u++) {
            const int32_t i = i0 + u * THREADS;
            if (i < ROWS * nA) {
                const int32_t row = i / nA;
                tile[(i - row * nA) * PITCH + row] = value[u];
            }
        }
    }
    if (tid < ROWS) {
        tile[nA * PITCH + tid] = T(0);
    }
}

/// Adds the terms of up to 64 table entries, the one of lane u being `coefficient` times the
/// values at byte offsets `place` of the tile, to the sums of the lane's rows; lanes from n on
/// hold entries that are zero, with places that exist.
template <typename T, int FACTORS, int RPL>
__device__ __forceinline__ void
add_terms(T (&sum)[RPL], const T* mine, T coefficient, const uint32_t (&place)[FACTORS > 0 ? FACTORS : 1], int32_t n) {
    constexpr int WORDS = sizeof(T) / 4;
    int32_t words[WORDS];
    __builtin_memcpy(words, &coefficient, sizeof(T));
    // BATCH entries at a time: first every LDS read, then the products (a read that is waited for
    // before the next one is asked for costs its whole latency)
    constexpr int BATCH = 8;
    for (int32_t u0 = 0; u0 < n; u0 += BATCH) {
        T term[BATCH];
        T value[BATCH][FACTORS > 0 ? FACTORS : 1][RPL];
#pragma unroll
        for (int b = 0; b < BATCH; b++) { // (u0 + b < 64: both are multiples of eight)
            int32_t uniform[WORDS];
#pragma unroll
            for (int w = 0; w < WORDS; w++) {
                uniform[w] = __builtin_amdgcn_readlane(words[w], u0 + b);
            }
            __builtin_memcpy(&term[b], uniform, sizeof(T));
#pragma unroll
            for (int k = 0; k < FACTORS; k++) {
                const uint32_t offset =
                    static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(place[k]), u0 + b));
                const T* at = reinterpret_cast<const T*>(reinterpret_cast<const char*>(mine) + offset);
#pragma unroll
                for (int r = 0; r < RPL; r++) {
                    value[b][k][r] = at[r * WAVE];
                }
            }
        }
#pragma unroll
        for (int b = 0; b < BATCH; b++) {
#pragma unroll
            for (int r = 0; r < RPL; r++) {
                T product = term[b];
#pragma unroll
                for (int k = 0; k < FACTORS; k++) {
                    product *= value[b][k][r];
                }
                sum[r] += product;
            }
        }
    }
}

// The wavefronts of a workgroup share the rows and take contiguous shares of the monomials; their
// partial sums meet in LDS in wave order. LDS: tile[nA + 1][pitch] partial[WAVES][rows]
template <typename T, int ORDER, int RPL>
__global__ __launch_bounds__(THREADS) void forward_kernel(
    T* __restrict__ output,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials
) {
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    constexpr int ROWS = rows_of(RPL), PITCH = pitch_of(RPL);
    T* tile = reinterpret_cast<T*>(lds_bytes);
    T* partial = tile + static_cast<size_t>(nA + 1) * PITCH;
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int32_t row0 = blockIdx.x * ROWS;
    const int32_t rows = min(ROWS, n_rows - row0);
    stage<T, RPL>(tile, A, row0, rows, nA);
    __syncthreads();

    const int32_t per_wave = (n_monomials + WAVES - 1) / WAVES;
    const int32_t begin = min(wave * per_wave, n_monomials);
    const int32_t end = min(begin + per_wave, n_monomials);
    T sum[RPL];
#pragma unroll
    for (int r = 0; r < RPL; r++) {
        sum[r] = T(0);
    }
    for (int32_t j0 = begin; j0 < end; j0 += WAVE) {
        const int32_t n = min(WAVE, end - j0);
        const int32_t j = lane < n ? j0 + lane : 0;
        const T coefficient = lane < n ? C[j] : T(0);
        uint32_t place[ORDER];
#pragma unroll
        for (int k = 0; k < ORDER; k++) {
            // (as unsigned, a negative index is a large one; beyond the last monomial: zeros)
            const uint32_t factor = static_cast<uint32_t>(P[static_cast<size_t>(j) * ORDER + k]);
            place[k] = min(lane < n ? factor : static_cast<uint32_t>(nA), static_cast<uint32_t>(nA)) *
                       static_cast<uint32_t>(PITCH * sizeof(T));
        }
        add_terms<T, ORDER, RPL>(sum, tile + lane, coefficient, place, n);
    }
#pragma unroll
    for (int r = 0; r < RPL; r++) {
        partial[wave * ROWS + lane + r * WAVE] = sum[r];
    }
    __syncthreads();
    if (tid < rows) {
        T total = T(0);
        for (int w = 0; w < WAVES; w++) {
            total += partial[w * ROWS + tid];
        }
        output[row0 + tid] = total;
    }
}

// A wavefront walks the terms of one feature's gradient at a time (hpe_tiles::TurnedTable);
// workgroup (x, y) has the features [y, y + 1) * features_per_group of its rows.
// LDS: tile[nA + 1][pitch] out[rows][out_pitch]
template <typename T, int ORDER, int RPL>
__global__ __launch_bounds__(THREADS) void vjp_kernel(
    T* __restrict__ grad_A,
    const T* __restrict__ grad_output,
    const T* __restrict__ A,
    const int32_t* __restrict__ lists,
    const uint32_t* __restrict__ records,
    int32_t n_rows,
    int32_t nA,
    int32_t features_per_group,
    int32_t out_pitch
) {
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    constexpr int ROWS = rows_of(RPL), PITCH = pitch_of(RPL);
    constexpr int OTHERS = ORDER - 1;
    constexpr int SIZE = OTHERS + static_cast<int>(sizeof(T) / 4);
    T* tile = reinterpret_cast<T*>(lds_bytes);
    T* out = tile + static_cast<size_t>(nA + 1) * PITCH;
    const int32_t first_feature = blockIdx.y * features_per_group;
    const int32_t n_features = min(features_per_group, nA - first_feature);
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int32_t row0 = blockIdx.x * ROWS;
    const int32_t rows = min(ROWS, n_rows - row0);
    stage<T, RPL>(tile, A, row0, rows, nA);
    T upstream[RPL];
#pragma unroll
    for (int r = 0; r < RPL; r++) {
        upstream[r] = load_or_zero(grad_output, static_cast<size_t>(row0 + lane + r * WAVE), lane + r * WAVE < rows);
    }
    __syncthreads();

    for (int32_t local = wave; local < n_features; local += WAVES) {
        const int32_t begin = lists[first_feature + local] * 4;
        const int32_t end = lists[first_feature + local + 1] * 4;
        T sum[RPL];
#pragma unroll
        for (int r = 0; r < RPL; r++) {
            sum[r] = T(0);
        }
        for (int32_t p0 = begin; p0 < end; p0 += WAVE) {
            const int32_t n = min(WAVE, end - p0);
            T coefficient = T(0);
            uint32_t place[OTHERS > 0 ? OTHERS : 1];
            const uint32_t* record = records + static_cast<size_t>(p0 + min(lane, n - 1)) * SIZE;
#pragma unroll
            for (int k = 0; k < OTHERS; k++) {
                place[k] = lane < n ? record[k] : static_cast<uint32_t>(nA) * static_cast<uint32_t>(PITCH * sizeof(T));
            }
            uint32_t words[sizeof(T) / 4];
#pragma unroll
            for (int w = 0; w < static_cast<int>(sizeof(T) / 4); w++) {
                words[w] = lane < n ? record[OTHERS + w] : 0u;
            }
            __builtin_memcpy(&coefficient, words, sizeof(T));
            add_terms<T, OTHERS, RPL>(sum, tile + lane, coefficient, place, n);
        }
#pragma unroll
        for (int r = 0; r < RPL; r++) {
            out[(lane + r * WAVE) * out_pitch + local] = upstream[r] * sum[r];
        }
    }
    __syncthreads();
    // row by row, this group's features next to each other (all of them: one contiguous piece)
    T* target = grad_A + static_cast<size_t>(row0) * nA + first_feature;
    for (int32_t i = tid; i < rows * n_features; i += THREADS) {
        const int32_t row = i / n_features;
        const int32_t local = i - row * n_features;
        target[static_cast<size_t>(row) * nA + local] = out[row * out_pitch + local];
    }
}

// --------------------------------------------------------------------- host --
size_t forward_lds(const Shape& s, int rpl, size_t element_size) {
    return ((static_cast<size_t>(s.nA) + 1) * pitch_of(rpl) + static_cast<size_t>(WAVES) * rows_of(rpl)) * element_size;
}
size_t vjp_lds(const Shape& s, int rpl, int32_t out_pitch, size_t element_size) {
    return ((static_cast<size_t>(s.nA) + 1) * pitch_of(rpl) + static_cast<size_t>(rows_of(rpl)) * out_pitch) * element_size;
}

/// How the vjp is cut: groups of 16 features (one per wavefront) while that brings the launch to a
/// few hundred workgroups, all features in one otherwise.
struct VjpPlan {
    int rows_per_lane;
    size_t row_groups;
    int32_t features_per_group;
    int32_t out_pitch;
    size_t lds;
};
VjpPlan plan_vjp(const Shape& s, size_t element_size) {
    VjpPlan plan;
    plan.rows_per_lane = vjp_lds(s, 2, (WAVES * 4) | 1, element_size) <= LDS_LIMIT ? 2 : 1;
    for (;; plan.rows_per_lane = 1) {
        plan.row_groups = ceil_div(static_cast<size_t>(s.n_rows), static_cast<size_t>(rows_of(plan.rows_per_lane)));
        const size_t wanted = std::max<size_t>(1, ceil_div(512, plan.row_groups));
        const size_t groups = std::min(wanted, ceil_div(static_cast<size_t>(s.nA), WAVES));
        plan.features_per_group =
            static_cast<int32_t>(ceil_div(ceil_div(static_cast<size_t>(s.nA), groups), WAVES) * WAVES);
        plan.out_pitch = plan.features_per_group | 1;
        plan.lds = vjp_lds(s, plan.rows_per_lane, plan.out_pitch, element_size);
        if (plan.lds <= LDS_LIMIT || plan.rows_per_lane == 1) {
            return plan;
        }
    }
}

template <typename Kernel> void allow_lds(Kernel kernel, size_t lds) {
    if (lds > 64 * 1024) {
        MOPS_HIP_CHECK(hipFuncSetAttribute(
            reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)
        ));
    }
}

template <typename Body> void with_order(int32_t order, Body&& body) {
    switch (order) {
    case 1:
        body(std::integral_constant<int, 1>{});
        break;
    case 2:
        body(std::integral_constant<int, 2>{});
        break;
    case 3:
        body(std::integral_constant<int, 3>{});
        break;
    case 4:
        body(std::integral_constant<int, 4>{});
        break;
    case 5:
        body(std::integral_constant<int, 5>{});
        break;
    default:
        body(std::integral_constant<int, 6>{});
        break;
    }
}

} // namespace

bool covers_forward(const Shape& s, size_t element_size) {
    return hpe_tiles::covered(s) && forward_lds(s, 1, element_size) <= LDS_LIMIT;
}

bool covers_vjp(const Shape& s, size_t element_size) {
    return hpe_tiles::covered(s) && s.nA <= hpe_tiles::MAX_FEATURES && plan_vjp(s, element_size).lds <= LDS_LIMIT;
}

template <typename T>
void forward(T* output, const T* A, const T* C, const int32_t* P, const Shape& s, hipStream_t stream) {
    const int rows_per_lane = forward_lds(s, 2, sizeof(T)) <= LDS_LIMIT ? 2 : 1;
    const size_t lds = forward_lds(s, rows_per_lane, sizeof(T));
    const unsigned blocks =
        static_cast<unsigned>(ceil_div(static_cast<size_t>(s.n_rows), static_cast<size_t>(rows_of(rows_per_lane))));
    with_order(s.order, [&](auto order) {
        constexpr int ORDER = decltype(order)::value;
        auto kernel = rows_per_lane == 2 ? forward_kernel<T, ORDER, 2> : forward_kernel<T, ORDER, 1>;
        allow_lds(kernel, lds);
        MainKernelTimer timer(stream);
        kernel<<<blocks, THREADS, lds, stream>>>(output, A, C, P, s.n_rows, s.nA, s.n_monomials);
    });
}

template <typename T>
void vjp(
    T* grad_A, const T* grad_output, const T* A, const T* C, const int32_t* P, const Shape& s, void* workspace,
    hipStream_t stream
) {
    const VjpPlan plan = plan_vjp(s, sizeof(T));
    const int32_t stride = pitch_of(plan.rows_per_lane) * static_cast<int32_t>(sizeof(T));
    const hpe_tiles::TurnedTable table = hpe_tiles::turn_table<T>(C, P, s, stride, workspace, stream);
    const dim3 blocks(
        static_cast<unsigned>(plan.row_groups),
        static_cast<unsigned>(ceil_div(static_cast<size_t>(s.nA), static_cast<size_t>(plan.features_per_group)))
    );
    with_order(s.order, [&](auto order) {
        constexpr int ORDER = decltype(order)::value;
        auto kernel = plan.rows_per_lane == 2 ? vjp_kernel<T, ORDER, 2> : vjp_kernel<T, ORDER, 1>;
        allow_lds(kernel, plan.lds);
        MainKernelTimer timer(stream);
        kernel<<<blocks, THREADS, plan.lds, stream>>>(
            grad_A, grad_output, A, table.lists, table.records, s.n_rows, s.nA, plan.features_per_group, plan.out_pitch
        );
    });
}

#define MOPS_INSTANTIATE(T)                                                                         \
    template void forward<T>(T*, const T*, const T*, const int32_t*, const Shape&, hipStream_t);   \
    template void vjp<T>(                                                                          \
        T*, const T*, const T*, const T*, const int32_t*, const Shape&, void*, hipStream_t         \
    );
MOPS_INSTANTIATE(float)
MOPS_INSTANTIATE(double)
#undef MOPS_INSTANTIATE

} // namespace hpe_rows
} // namespace mops::amd
