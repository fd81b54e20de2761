// Homogeneous polynomial evaluation (HPE), forward and vector-Jacobian
// product, for gfx950.
//
//   O[i] = sum_j C[j] * prod_k A[i, P[j, k]]
//   grad_A[i, P[j, f]] += C[j] * grad_O[i] * prod_{k != f} A[i, P[j, k]]
//
// Semantics restated from mops/src/hpe/cpu.tpp:13-272 of lab-cosmo/mops:
// each monomial's product starts from C[j] and multiplies the factors left
// to right; a polynomial of order 0 gives O[i] = sum_j C[j]; the vjp is a
// no-op when grad_A is not requested. (The CPU reference stops at order 10;
// there is no such limit here.)
//
// Work split: a workgroup takes `R` consecutive batch rows (R a power of two,
// 1..64) and G = blockDim / R monomial groups; thread (r, g) evaluates the
// monomials j = g, g + G, ... for row r. The rows' A values sit in LDS as
// [feature][row]. Small batches get R = 1 (the whole workgroup shares one row
// and spreads over the monomials), large batches R = 64 (one row per lane,
// the table read once per wavefront), so that there are always enough
// workgroups to fill the device.
//
// The partial sums of the G groups are combined in group order, so results
// are reproducible from run to run. The reference's CUDA vjp accumulates
// with shared-memory float atomics (mops/src/hpe/hpe.cu:288) and is not.
#include <algorithm>
#include <type_traits>

#include "mops/hpe.hpp"

#include "checks.hpp"
#include "device_common.hpp"
#include "dispatch_thresholds.hpp"
#include "index_validation.hpp"
#include "elementwise.hpp"
#include "hpe_rows.hpp"
#include "hpe_tiles.hpp"
#include "runtime.hpp"

namespace mops::amd {
namespace hpe { // a name of its own for this file's kernels: profilers print it
namespace {

constexpr size_t LDS_BUDGET = 60 * 1024;

// ---------------------------------------------------------------------------
// forward. LDS: a[nA][R] partial[G][R]
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void forward_kernel(
    T* __restrict__ output,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials,
    int32_t order,
    int32_t R
) {
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    T* a_stage = reinterpret_cast<T*>(lds_bytes);
    T* partial = a_stage + static_cast<size_t>(nA) * R;

    const int tid = threadIdx.x;
    const int G = blockDim.x / R;
    const int r = tid % R;
    const int g = tid / R;
    const int32_t row0 = blockIdx.x * R;
    const int32_t rows = min(R, n_rows - row0);

    const T* a_src = A + static_cast<size_t>(row0) * nA;
    for (int32_t i = tid; i < rows * nA; i += blockDim.x) {
        int32_t row = i / nA;
        a_stage[(i - row * nA) * R + row] = a_src[i];
    }
    __syncthreads();

    T sum = T(0);
    if (r < rows) {
        for (int32_t j = g; j < n_monomials; j += G) {
            const int32_t* factors = P + static_cast<size_t>(j) * order;
            T product = C[j];
            for (int32_t k = 0; k < order; k++) {
                int32_t feature = factors[k];
                product *= in_bounds(feature, nA) ? a_stage[feature * R + r] : T(0);
            }
            sum += product;
        }
    }
    partial[g * R + r] = sum;
    __syncthreads();
    if (g == 0 && r < rows) {
        T total = T(0);
        for (int group = 0; group < G; group++) {
            total += partial[group * R + r];
        }
        output[row0 + r] = total;
    }
}

// ---------------------------------------------------------------------------
// forward with the order known at compile time: factors and the values they
// select in registers, the next monomial fetched while the current one is
// multiplied, and the partial sums of the groups combined by a fixed tree
// (shuffles inside a wavefront, then the wavefronts in order) instead of one
// thread walking over all of them. R is a power of two.
// ---------------------------------------------------------------------------
template <typename T, int ORDER>
__global__ __launch_bounds__(256) void forward_ordered_kernel(
    T* __restrict__ output,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials,
    int32_t R
) {
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    // a[nA + 1][R]: the row after the last stays zero, a factor outside [0, nA)
    // reads it, and the loop over the monomials has no branch in it
    T* a_stage = reinterpret_cast<T*>(lds_bytes);
    T* partial = a_stage + static_cast<size_t>(nA + 1) * R;

    const int tid = threadIdx.x;
    const int G = blockDim.x / R;
    const int r = tid % R;
    const int g = tid / R;
    const int32_t row0 = blockIdx.x * R;
    const int32_t rows = min(R, n_rows - row0);

    const T* a_src = A + static_cast<size_t>(row0) * nA;
    for (int32_t i = tid; i < rows * nA; i += blockDim.x) {
        int32_t row = i / nA;
        a_stage[(i - row * nA) * R + row] = a_src[i];
    }
    if (tid < R) {
        a_stage[nA * R + tid] = T(0);
    }
    __syncthreads();

    struct Monomial {
        int32_t factor[ORDER > 0 ? ORDER : 1];
        T coefficient;
    };
    auto fetch = [&](Monomial& to, int32_t j) {
        const int32_t safe = min(j, n_monomials - 1);
        const int32_t* factors = P + static_cast<size_t>(safe) * ORDER;
#pragma unroll
        for (int k = 0; k < ORDER; k++) {
            to.factor[k] = factors[k];
        }
        to.coefficient = C[safe];
    };
    // BATCH monomials at a time: their factors asked for together, then their
    // values of A, then the products (independent chains); a monomial beyond
    // the last counts with coefficient zero.
    T sum = T(0);
    if (r < rows && n_monomials > 0) {
        constexpr int BATCH = 4;
        const uint32_t features = static_cast<uint32_t>(nA);
        const T* my_a = a_stage + r;
        Monomial next[BATCH];
#pragma unroll
        for (int d = 0; d < BATCH; d++) {
            fetch(next[d], g + d * G);
        }
        for (int32_t j0 = g; j0 < n_monomials; j0 += BATCH * G) {
            Monomial now[BATCH];
            T value[BATCH][ORDER > 0 ? ORDER : 1];
#pragma unroll
            for (int d = 0; d < BATCH; d++) {
                now[d] = next[d];
#pragma unroll
                for (int k = 0; k < ORDER; k++) {
                    // (as unsigned, a negative factor is a large one)
                    value[d][k] = my_a[min(static_cast<uint32_t>(now[d].factor[k]), features) * R];
                }
            }
#pragma unroll
            for (int d = 0; d < BATCH; d++) {
                fetch(next[d], j0 + (d + BATCH) * G);
            }
#pragma unroll
            for (int d = 0; d < BATCH; d++) {
                T product = j0 + d * G < n_monomials ? now[d].coefficient : T(0);
#pragma unroll
                for (int k = 0; k < ORDER; k++) {
                    product *= value[d][k];
                }
                sum += product;
            }
        }
    }
    // lanes with the same r inside a wavefront, then the wavefronts
    for (int offset = WAVE / 2; offset >= R; offset >>= 1) {
        sum += __shfl_xor(sum, offset);
    }
    const int wave = tid / WAVE;
    const int lane = tid % WAVE;
    if (R <= WAVE) {
        if (lane < R) {
            partial[wave * R + lane] = sum;
        }
    } else {
        partial[g * R + r] = sum;
    }
    __syncthreads();
    const int copies = R <= WAVE ? static_cast<int>(blockDim.x) / WAVE : G;
    if (tid < rows) {
        T total = T(0);
        for (int copy = 0; copy < copies; copy++) {
            total += partial[copy * R + tid];
        }
        output[row0 + tid] = total;
    }
}

// ---------------------------------------------------------------------------
// vjp. One wavefront per workgroup. LDS: a[nA][R] accumulator[G][span][R]
// Thread (r, g) adds its monomials' terms into its private accumulator row
// set; afterwards the G copies are added in group order.
// `span` = nA when the accumulators of all features fit in LDS; otherwise the
// features are split into ranges of `span`, blockIdx.y picks the range, and a
// workgroup walks all monomials but keeps only the terms for its range.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(WAVE) void vjp_kernel(
    T* __restrict__ grad_A,
    const T* __restrict__ grad_output,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials,
    int32_t order,
    int32_t R,
    int32_t span
) {
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    T* a_stage = reinterpret_cast<T*>(lds_bytes);
    T* accumulator = a_stage + static_cast<size_t>(nA) * R;
    const int32_t feature_begin = blockIdx.y * span;
    const int32_t feature_count = min(span, nA - feature_begin);

    const int tid = threadIdx.x;
    const int G = WAVE / R;
    const int r = tid % R;
    const int g = tid / R;
    const int32_t row0 = blockIdx.x * R;
    const int32_t rows = min(R, n_rows - row0);

    const T* a_src = A + static_cast<size_t>(row0) * nA;
    for (int32_t i = tid; i < rows * nA; i += WAVE) {
        int32_t row = i / nA;
        a_stage[(i - row * nA) * R + row] = a_src[i];
    }
    for (int32_t i = tid; i < G * feature_count * R; i += WAVE) {
        accumulator[i] = T(0);
    }
    __syncthreads();

    if (r < rows) {
        T* mine = accumulator + static_cast<size_t>(g) * feature_count * R + r;
        const T upstream = grad_output[row0 + r];
        for (int32_t j = g; j < n_monomials; j += G) {
            const int32_t* factors = P + static_cast<size_t>(j) * order;
            const T base = C[j] * upstream;
            for (int32_t f = 0; f < order; f++) {
                int32_t target = factors[f] - feature_begin;
                if (!in_bounds(target, feature_count)) {
                    continue;
                }
                T term = base;
                for (int32_t k = 0; k < order; k++) {
                    if (k == f) {
                        continue;
                    }
                    int32_t feature = factors[k];
                    term *= in_bounds(feature, nA) ? a_stage[feature * R + r] : T(0);
                }
                mine[target * R] += term;
            }
        }
    }
    __syncthreads();

    T* dst = grad_A + static_cast<size_t>(row0) * nA + feature_begin;
    for (int32_t i = tid; i < rows * feature_count; i += WAVE) {
        int32_t row = i / feature_count;
        int32_t feature = i - row * feature_count;
        T total = T(0);
        for (int group = 0; group < G; group++) {
            total += accumulator[(static_cast<size_t>(group) * feature_count + feature) * R + row];
        }
        dst[static_cast<size_t>(row) * nA + feature] = total;
    }
}

// ---------------------------------------------------------------------------
// vjp with the order known at compile time: same layout as vjp_kernel, but a
// monomial's factors, the values they select and the K partial products
// (prefix * suffix, 3 K multiplications instead of K^2) live in registers, and
// the factors of the next monomial are fetched while the current one is used.
// ---------------------------------------------------------------------------
constexpr int ORDERED_VJP_THREADS = 4 * WAVE; // one wavefront that walks the monomials and three helpers

template <typename T, int ORDER>
__global__ __launch_bounds__(ORDERED_VJP_THREADS) void vjp_ordered_kernel(
    T* __restrict__ grad_A,
    const T* __restrict__ grad_output,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials,
    int32_t log2_R
) {
    // LDS: a[nA + 1][R] accumulator[G][nA + 1][R]. The extra row of `a` stays zero
    // and the extra accumulator row is never read: a factor outside [0, nA)
    // reads the one, its term and those of a monomial beyond the last go to the
    // other, and the loop over the monomials has no branch in it.
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    const int32_t R = 1 << log2_R;
    T* a_stage = reinterpret_cast<T*>(lds_bytes);
    T* accumulator = a_stage + static_cast<size_t>(nA + 1) * R;

    // Thread (r, g) of the FIRST wavefront walks the monomials; the other
    // wavefronts of the workgroup only help to stage the rows, to clear the
    // accumulators and to add up the copies, which a single wavefront would
    // spend a third of the launch on.
    const int tid = threadIdx.x;
    const bool walks = tid < WAVE;
    const int G = WAVE >> log2_R;
    const int r = tid & (R - 1);
    const int g = (tid & (WAVE - 1)) >> log2_R;
    const int32_t row0 = blockIdx.x * R;
    const int32_t rows = min(R, n_rows - row0);

    struct Monomial {
        int32_t factor[ORDER];
        T coefficient;
    };
    auto fetch = [&](Monomial& to, int32_t j) {
        const int32_t safe = min(j, n_monomials - 1);
        const int32_t* factors = P + static_cast<size_t>(safe) * ORDER;
#pragma unroll
        for (int k = 0; k < ORDER; k++) {
            to.factor[k] = factors[k];
        }
        to.coefficient = C[safe];
    };
    // A compute unit holds three of these wavefronts (their accumulators fill
    // its LDS), so nobody else covers a thread's waits and every instruction
    // counts. A thread works on BATCH monomials at a time, in three phases:
    // all their values of A are asked for from LDS together, then all their
    // terms are multiplied up in registers (BATCH independent chains), then
    // all terms are added to the accumulators, in the order of the
    // monomials. The factors of the next batch are on their way from global
    // memory meanwhile, those of the first one while the tiles are set up.
    constexpr int BATCH = 8;
    Monomial queue[BATCH];
    T upstream = T(0);
    if (walks) {
#pragma unroll
        for (int d = 0; d < BATCH; d++) {
            fetch(queue[d], g + d * G);
        }
        upstream = grad_output[min(row0 + r, n_rows - 1)];
    }

    // the rows of A, STAGE values per lane asked for together: with one load
    // per turn of a loop, each turn would wait a whole round trip to memory
    const T* a_src = A + static_cast<size_t>(row0) * nA;
    constexpr int STAGE = 8;
    for (int32_t base = 0; base < rows * nA; base += STAGE * ORDERED_VJP_THREADS) {
        T staged[STAGE];
#pragma unroll
        for (int u = 0; u < STAGE; u++) {
            const int32_t i = base + u * ORDERED_VJP_THREADS + tid;
            staged[u] = a_src[min(i, rows * nA - 1)];
        }
#pragma unroll
        for (int u = 0; u < STAGE; u++) {
            const int32_t i = base + u * ORDERED_VJP_THREADS + tid;
            if (i < rows * nA) {
                const int32_t row = i / nA;
                a_stage[((i - row * nA) << log2_R) + row] = staged[u];
            }
        }
    }
    if (tid < R) {
        a_stage[nA * R + tid] = T(0);
    }
    // (G * R = 64: the accumulators are nA + 1 rows of 64 values, one
    // per lane; wavefront w clears rows w, w + 4, ...; unrolled, because a
    // wavefront pays for every instruction of the loop around a store)
    {
        constexpr int HELPERS = ORDERED_VJP_THREADS / WAVE;
        T* clear = accumulator + (tid & (WAVE - 1));
        int32_t k = tid >> 6;
        for (; k + 7 * HELPERS < nA + 1; k += 8 * HELPERS) {
#pragma unroll
            for (int u = 0; u < 8; u++) {
                clear[(k + u * HELPERS) * WAVE] = T(0);
            }
        }
        for (; k < nA + 1; k += HELPERS) {
            clear[k * WAVE] = T(0);
        }
    }
    __syncthreads();

    if (walks && r < rows) {
        T* mine = accumulator + static_cast<size_t>(g) * (nA + 1) * R + r;
        const T* my_a = a_stage + r;
        // a feature's distance in bytes as a shift: address = base + (feature << shift), one
        // instruction (shift-and-add) per LDS access instead of a shift, a scaling and an add
        const int32_t byte_shift = log2_R + (sizeof(T) == 8 ? 3 : 2);
        auto at = [&](auto* base, uint32_t feature) {
            using Pointer = decltype(base);
            using Bytes = std::conditional_t<std::is_const_v<std::remove_pointer_t<Pointer>>, const char*, char*>;
            return reinterpret_cast<Pointer>(reinterpret_cast<Bytes>(base) + (feature << byte_shift));
        };
        const uint32_t features = static_cast<uint32_t>(nA);
        // `whole`: all monomials of the batch exist
        auto batch = [&](int32_t j0, auto whole) {
            constexpr bool WHOLE = decltype(whole)::value;
            Monomial now[BATCH];
            T value[BATCH][ORDER];
#pragma unroll
            for (int d = 0; d < BATCH; d++) {
                now[d] = queue[d];
#pragma unroll
                for (int k = 0; k < ORDER; k++) {
                    // (as unsigned, a negative factor is a large one)
                    const uint32_t feature = min(static_cast<uint32_t>(now[d].factor[k]), features);
                    value[d][k] = *at(my_a, feature);
                }
            }
            if constexpr (WHOLE) {
#pragma unroll
                for (int d = 0; d < BATCH; d++) {
                    fetch(queue[d], j0 + (d + BATCH) * G);
                }
            }
            // term[f] = base * prod_{k != f} value[k], multiplied left to right
            T term[BATCH][ORDER];
#pragma unroll
            for (int d = 0; d < BATCH; d++) {
                T prefix[ORDER];
                prefix[0] = now[d].coefficient * upstream;
#pragma unroll
                for (int k = 1; k < ORDER; k++) {
                    prefix[k] = prefix[k - 1] * value[d][k - 1];
                }
                T suffix = T(1);
#pragma unroll
                for (int f = ORDER - 1; f >= 0; f--) {
                    term[d][f] = prefix[f] * suffix;
                    suffix *= value[d][f];
                }
            }
#pragma unroll
            for (int d = 0; d < BATCH; d++) {
                const bool exists = WHOLE || j0 + d * G < n_monomials;
#pragma unroll
                for (int f = ORDER - 1; f >= 0; f--) {
                    const uint32_t slot = min(static_cast<uint32_t>(now[d].factor[f]), features);
                    T* to = at(mine, exists ? slot : features);
                    // a slot of my own. In f64 the LDS add instruction, which saves the
                    // round trip of read, add, write; in f32 that instruction is the
                    // slower way here (53 us against 21)
                    if constexpr (sizeof(T) == 8) {
                        unsafeAtomicAdd(to, term[d][f]);
                    } else {
                        *to += term[d][f];
                    }
                }
            }
        };
        int32_t j0 = g;
        for (; j0 + (BATCH - 1) * G < n_monomials; j0 += BATCH * G) {
            batch(j0, std::true_type{});
        }
        if (j0 < n_monomials) {
            batch(j0, std::false_type{});
        }
    }
    __syncthreads();

    // The G copies added up, every (feature, row) by one lane: four running
    // sums over the copies g = 0, 4, ... / 1, 5, ... / 2, 6, ... / 3, 7, ...
    // and then (s0 + s1) + (s2 + s3): one fixed order, and chains of additions
    // a quarter as long as one sum over all copies would be.
    T* dst = grad_A + static_cast<size_t>(row0) * nA;
    const int32_t copy_stride = (nA + 1) * R;
    for (int32_t entry = tid; entry < nA * R; entry += ORDERED_VJP_THREADS) {
        const int32_t row = entry & (R - 1);
        const int32_t feature = entry >> log2_R;
        const T* from = accumulator + entry;
        T partial[4] = {T(0), T(0), T(0), T(0)};
        int group = 0;
        for (; group + 4 <= G; group += 4) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                partial[u] += from[(group + u) * copy_stride];
            }
        }
        for (; group < G; group++) {
            partial[group & 3] += from[group * copy_stride];
        }
        if (row < rows) {
            dst[static_cast<size_t>(row) * nA + feature] = (partial[0] + partial[1]) + (partial[2] + partial[3]);
        }
    }
}

// ---------------------------------------------------------------------------
// Fallbacks for feature counts whose tiles do not fit in LDS: one thread per
// batch row, everything in global memory.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void forward_global_kernel(
    T* __restrict__ output,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials,
    int32_t order
) {
    const int32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= n_rows) {
        return;
    }
    const T* a_row = A + static_cast<size_t>(row) * nA;
    T sum = T(0);
    for (int32_t j = 0; j < n_monomials; j++) {
        const int32_t* factors = P + static_cast<size_t>(j) * order;
        T product = C[j];
        for (int32_t k = 0; k < order; k++) {
            int32_t feature = factors[k];
            product *= in_bounds(feature, nA) ? a_row[feature] : T(0);
        }
        sum += product;
    }
    output[row] = sum;
}

template <typename T>
__global__ __launch_bounds__(256) void vjp_global_kernel(
    T* grad_A,
    const T* __restrict__ grad_output,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials,
    int32_t order
) {
    const int32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= n_rows) {
        return;
    }
    const T* a_row = A + static_cast<size_t>(row) * nA;
    T* g_row = grad_A + static_cast<size_t>(row) * nA;
    for (int32_t feature = 0; feature < nA; feature++) {
        g_row[feature] = T(0);
    }
    const T upstream = grad_output[row];
    for (int32_t j = 0; j < n_monomials; j++) {
        const int32_t* factors = P + static_cast<size_t>(j) * order;
        const T base = C[j] * upstream;
        for (int32_t f = 0; f < order; f++) {
            int32_t target = factors[f];
            if (!in_bounds(target, nA)) {
                continue;
            }
            T term = base;
            for (int32_t k = 0; k < order; k++) {
                if (k == f) {
                    continue;
                }
                int32_t feature = factors[k];
                term *= in_bounds(feature, nA) ? a_row[feature] : T(0);
            }
            g_row[target] += term;
        }
    }
}

// ---------------------------------------------------------------------------
// Second order: the vjp of the vjp (semantics of mops/src/hpe/cpu.tpp:275-539).
//
//   grad_grad_O[i]      = sum_j C[j] sum_f gg[i, P[j, f]] prod_{k != f} A[i, P[j, k]]
//   grad_A_2[i, P[j,f2]] += gO[i] C[j] sum_{f != f2} gg[i, P[j, f]] prod_{k != f, f2} A[i, P[j, k]]
//
// with gg = grad_grad_A. Same work split as vjp_kernel: one wavefront per
// workgroup, thread (r, g) walks the monomials j = g, g + G, ... of row r and
// adds into private accumulators in LDS, which are then combined in group
// order. LDS: a[nA][R] gg[nA][R] accumulator[G][nA][R] partial[G][R].
// Either output may be null.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(WAVE) void vjp_vjp_kernel(
    T* __restrict__ grad_grad_output,
    T* __restrict__ grad_A_2,
    const T* __restrict__ grad_grad_A,
    const T* __restrict__ grad_output,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials,
    int32_t order,
    int32_t R
) {
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    T* a_stage = reinterpret_cast<T*>(lds_bytes);
    T* gg_stage = a_stage + static_cast<size_t>(nA) * R;
    T* accumulator = gg_stage + static_cast<size_t>(nA) * R;
    T* partial = accumulator + static_cast<size_t>(nA) * WAVE;

    const int tid = threadIdx.x;
    const int G = WAVE / R;
    const int r = tid % R;
    const int g = tid / R;
    const int32_t row0 = blockIdx.x * R;
    const int32_t rows = min(R, n_rows - row0);
    const bool want_O = grad_grad_output != nullptr;
    const bool want_A = grad_A_2 != nullptr;

    const T* a_src = A + static_cast<size_t>(row0) * nA;
    const T* gg_src = grad_grad_A + static_cast<size_t>(row0) * nA;
    for (int32_t i = tid; i < rows * nA; i += WAVE) {
        const int32_t row = i / nA;
        a_stage[(i - row * nA) * R + row] = a_src[i];
        gg_stage[(i - row * nA) * R + row] = gg_src[i];
    }
    for (int32_t i = tid; i < nA * WAVE; i += WAVE) {
        accumulator[i] = T(0);
    }
    __syncthreads();

    T sum = T(0);
    if (r < rows) {
        T* mine = accumulator + static_cast<size_t>(g) * nA * R + r;
        const T upstream = grad_output[row0 + r];
        auto value_of = [&](const T* stage, int32_t feature) {
            return in_bounds(feature, nA) ? stage[feature * R + r] : T(0);
        };
        for (int32_t j = g; j < n_monomials; j += G) {
            const int32_t* factors = P + static_cast<size_t>(j) * order;
            const T coefficient = C[j];
            if (want_O) {
                for (int32_t f = 0; f < order; f++) {
                    T term = coefficient * value_of(gg_stage, factors[f]);
                    for (int32_t k = 0; k < order; k++) {
                        if (k != f) {
                            term *= value_of(a_stage, factors[k]);
                        }
                    }
                    sum += term;
                }
            }
            if (want_A) {
                const T base = coefficient * upstream;
                for (int32_t f2 = 0; f2 < order; f2++) {
                    const int32_t target = factors[f2];
                    if (!in_bounds(target, nA)) {
                        continue;
                    }
                    T total = T(0);
                    for (int32_t f = 0; f < order; f++) {
                        if (f == f2) {
                            continue;
                        }
                        T term = base * value_of(gg_stage, factors[f]);
                        for (int32_t k = 0; k < order; k++) {
                            if (k != f && k != f2) {
                                term *= value_of(a_stage, factors[k]);
                            }
                        }
                        total += term;
                    }
                    mine[target * R] += total;
                }
            }
        }
    }
    partial[g * R + r] = sum;
    __syncthreads();

    if (want_O && tid < rows) {
        T total = T(0);
        for (int group = 0; group < G; group++) {
            total += partial[group * R + tid];
        }
        grad_grad_output[row0 + tid] = total;
    }
    if (want_A) {
        T* dst = grad_A_2 + static_cast<size_t>(row0) * nA;
        for (int32_t i = tid; i < rows * nA; i += WAVE) {
            const int32_t row = i / nA;
            const int32_t feature = i - row * nA;
            T total = T(0);
            for (int group = 0; group < G; group++) {
                total += accumulator[(static_cast<size_t>(group) * nA + feature) * R + row];
            }
            dst[i] = total;
        }
    }
}

// ---------------------------------------------------------------------------
// Second order with the order known at compile time. Layout and division of
// labour of vjp_ordered_kernel (the first wavefront walks the monomials, the
// others help to stage, clear and add up), with a tile of grad_grad_A beside
// the tile of A. A monomial costs O(K) instead of O(K^3): with a = A[i, P[j, .]]
// and g = grad_grad_A[i, P[j, .]], the sums above are the derivative of the
// product of the a's along g and that derivative's gradient,
//
//   S      = sum_f g[f] prod_{k != f} a[k]              (into grad_grad_output)
//   D[f2]  = sum_{f != f2} g[f] prod_{k != f, f2} a[k]   (into grad_A_2, times gO)
//
// and both come from products of the factors before and after a position that
// carry their own derivative along g:  p' = p a,  dp' = dp a + p g.
// Then D[f2] = dp[f2] s[f2] + p[f2] ds[f2] and S = dp[K].
// LDS: a[nA + 1][R] gg[nA + 1][R] accumulator[G][nA + 1][R]
// ---------------------------------------------------------------------------
template <typename T, int ORDER>
__global__ __launch_bounds__(ORDERED_VJP_THREADS) void vjp_vjp_ordered_kernel(
    T* __restrict__ grad_grad_output,
    T* __restrict__ grad_A_2,
    const T* __restrict__ grad_grad_A,
    const T* __restrict__ grad_output,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials,
    int32_t log2_R
) {
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    const int32_t R = 1 << log2_R;
    T* a_stage = reinterpret_cast<T*>(lds_bytes);
    T* gg_stage = a_stage + static_cast<size_t>(nA + 1) * R;
    T* accumulator = gg_stage + static_cast<size_t>(nA + 1) * R;
    const bool want_O = grad_grad_output != nullptr;
    const bool want_A = grad_A_2 != nullptr;

    const int tid = threadIdx.x;
    const bool walks = tid < WAVE;
    const int G = WAVE >> log2_R;
    const int r = tid & (R - 1);
    const int g = (tid & (WAVE - 1)) >> log2_R;
    const int32_t row0 = blockIdx.x * R;
    const int32_t rows = min(R, n_rows - row0);

    struct Monomial {
        int32_t factor[ORDER];
        T coefficient;
    };
    auto fetch = [&](Monomial& to, int32_t j) {
        const int32_t safe = min(j, n_monomials - 1);
        const int32_t* factors = P + static_cast<size_t>(safe) * ORDER;
#pragma unroll
        for (int k = 0; k < ORDER; k++) {
            to.factor[k] = factors[k];
        }
        to.coefficient = C[safe];
    };
    constexpr int BATCH = 4;
    Monomial queue[BATCH];
    T upstream = T(0);
    if (walks) {
#pragma unroll
        for (int d = 0; d < BATCH; d++) {
            fetch(queue[d], g + d * G);
        }
        upstream = grad_output[min(row0 + r, n_rows - 1)];
    }

    // the rows of A and of grad_grad_A, STAGE values of each per lane asked for together
    const T* a_src = A + static_cast<size_t>(row0) * nA;
    const T* gg_src = grad_grad_A + static_cast<size_t>(row0) * nA;
    constexpr int STAGE = 4;
    for (int32_t base = 0; base < rows * nA; base += STAGE * ORDERED_VJP_THREADS) {
        T staged[2][STAGE];
#pragma unroll
        for (int u = 0; u < STAGE; u++) {
            const int32_t i = min(base + u * ORDERED_VJP_THREADS + tid, rows * nA - 1);
            staged[0][u] = a_src[i];
            staged[1][u] = gg_src[i];
        }
#pragma unroll
        for (int u = 0; u < STAGE; u++) {
            const int32_t i = base + u * ORDERED_VJP_THREADS + tid;
            if (i < rows * nA) {
                const int32_t row = i / nA;
                const int32_t at = ((i - row * nA) << log2_R) + row;
                a_stage[at] = staged[0][u];
                gg_stage[at] = staged[1][u];
            }
        }
    }
    if (tid < R) {
        a_stage[nA * R + tid] = T(0);
        gg_stage[nA * R + tid] = T(0);
    }
    if (want_A) {
        constexpr int HELPERS = ORDERED_VJP_THREADS / WAVE;
        T* clear = accumulator + (tid & (WAVE - 1));
        int32_t k = tid >> 6;
        for (; k + 7 * HELPERS < nA + 1; k += 8 * HELPERS) {
#pragma unroll
            for (int u = 0; u < 8; u++) {
                clear[(k + u * HELPERS) * WAVE] = T(0);
            }
        }
        for (; k < nA + 1; k += HELPERS) {
            clear[k * WAVE] = T(0);
        }
    }
    __syncthreads();

    T sum = T(0);
    if (walks && r < rows) {
        T* mine = accumulator + static_cast<size_t>(g) * (nA + 1) * R + r;
        const int32_t byte_shift = log2_R + (sizeof(T) == 8 ? 3 : 2);
        auto at = [&](auto* base, uint32_t feature) {
            using Pointer = decltype(base);
            using Bytes = std::conditional_t<std::is_const_v<std::remove_pointer_t<Pointer>>, const char*, char*>;
            return reinterpret_cast<Pointer>(reinterpret_cast<Bytes>(base) + (feature << byte_shift));
        };
        const T* my_a = a_stage + r;
        const T* my_gg = gg_stage + r;
        const uint32_t features = static_cast<uint32_t>(nA);
        auto batch = [&](int32_t j0, auto whole) {
            constexpr bool WHOLE = decltype(whole)::value;
            Monomial now[BATCH];
            T a[BATCH][ORDER];
            T gg[BATCH][ORDER];
#pragma unroll
            for (int d = 0; d < BATCH; d++) {
                now[d] = queue[d];
#pragma unroll
                for (int k = 0; k < ORDER; k++) {
                    // (as unsigned, a negative factor is a large one)
                    const uint32_t feature = min(static_cast<uint32_t>(now[d].factor[k]), features);
                    a[d][k] = *at(my_a, feature);
                    gg[d][k] = *at(my_gg, feature);
                }
            }
            if constexpr (WHOLE) {
#pragma unroll
                for (int d = 0; d < BATCH; d++) {
                    fetch(queue[d], j0 + (d + BATCH) * G);
                }
            }
            T term[BATCH][ORDER];
#pragma unroll
            for (int d = 0; d < BATCH; d++) {
                const bool exists = WHOLE || j0 + d * G < n_monomials;
                // products of the factors before a position, and their derivative along gg
                T before[ORDER + 1];
                T d_before[ORDER + 1];
                before[0] = exists ? now[d].coefficient : T(0);
                d_before[0] = T(0);
#pragma unroll
                for (int k = 0; k < ORDER; k++) {
                    before[k + 1] = before[k] * a[d][k];
                    d_before[k + 1] = d_before[k] * a[d][k] + before[k] * gg[d][k];
                }
                sum += d_before[ORDER];
                // the same from the other end, and the two put together
                T after = T(1);
                T d_after = T(0);
#pragma unroll
                for (int f = ORDER - 1; f >= 0; f--) {
                    term[d][f] = upstream * (d_before[f] * after + before[f] * d_after);
                    d_after = d_after * a[d][f] + after * gg[d][f];
                    after *= a[d][f];
                }
            }
            if (want_A) {
#pragma unroll
                for (int d = 0; d < BATCH; d++) {
#pragma unroll
                    for (int f = ORDER - 1; f >= 0; f--) {
                        // (a factor outside [0, nA) and a monomial beyond the last, whose terms
                        // are zero, go to the row that is never read)
                        T* to = at(mine, min(static_cast<uint32_t>(now[d].factor[f]), features));
                        if constexpr (sizeof(T) == 8) {
                            unsafeAtomicAdd(to, term[d][f]);
                        } else {
                            *to += term[d][f];
                        }
                    }
                }
            }
        };
        int32_t j0 = g;
        for (; j0 + (BATCH - 1) * G < n_monomials; j0 += BATCH * G) {
            batch(j0, std::true_type{});
        }
        if (j0 < n_monomials) {
            batch(j0, std::false_type{});
        }
    }
    // grad_grad_output: the lanes of the first wavefront that share a row, by a fixed tree
    if (walks && want_O) {
        for (int offset = WAVE / 2; offset >= R; offset >>= 1) {
            sum += __shfl_xor(sum, offset);
        }
        if (tid < rows) {
            grad_grad_output[row0 + tid] = sum;
        }
    }
    __syncthreads();

    if (want_A) {
        T* dst = grad_A_2 + static_cast<size_t>(row0) * nA;
        const int32_t copy_stride = (nA + 1) * R;
        for (int32_t entry = tid; entry < nA * R; entry += ORDERED_VJP_THREADS) {
            const int32_t row = entry & (R - 1);
            const int32_t feature = entry >> log2_R;
            const T* from = accumulator + entry;
            T partial[4] = {T(0), T(0), T(0), T(0)};
            int group = 0;
            for (; group + 4 <= G; group += 4) {
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    partial[u] += from[(group + u) * copy_stride];
                }
            }
            for (; group < G; group++) {
                partial[group & 3] += from[group * copy_stride];
            }
            if (row < rows) {
                dst[static_cast<size_t>(row) * nA + feature] = (partial[0] + partial[1]) + (partial[2] + partial[3]);
            }
        }
    }
}

// The same with everything in global memory, one thread per batch row, for
// feature counts whose tiles do not fit in LDS.
template <typename T>
__global__ __launch_bounds__(256) void vjp_vjp_global_kernel(
    T* grad_grad_output,
    T* grad_A_2,
    const T* __restrict__ grad_grad_A,
    const T* __restrict__ grad_output,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials,
    int32_t order
) {
    const int32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= n_rows) {
        return;
    }
    const T* a_row = A + static_cast<size_t>(row) * nA;
    const T* gg_row = grad_grad_A + static_cast<size_t>(row) * nA;
    T* out_row = grad_A_2 != nullptr ? grad_A_2 + static_cast<size_t>(row) * nA : nullptr;
    if (out_row != nullptr) {
        for (int32_t feature = 0; feature < nA; feature++) {
            out_row[feature] = T(0);
        }
    }
    auto value_of = [&](const T* values, int32_t feature) {
        return in_bounds(feature, nA) ? values[feature] : T(0);
    };
    const T upstream = grad_output[row];
    T sum = T(0);
    for (int32_t j = 0; j < n_monomials; j++) {
        const int32_t* factors = P + static_cast<size_t>(j) * order;
        for (int32_t f2 = 0; f2 < order; f2++) {
            // f2 = the factor differentiated last; the f2-th term of the first
            // sum is the product with gg in place of that factor
            T first = C[j] * value_of(gg_row, factors[f2]);
            T second = T(0);
            for (int32_t k = 0; k < order; k++) {
                if (k != f2) {
                    first *= value_of(a_row, factors[k]);
                }
            }
            sum += first;
            if (out_row != nullptr && in_bounds(factors[f2], nA)) {
                for (int32_t f = 0; f < order; f++) {
                    if (f == f2) {
                        continue;
                    }
                    T term = C[j] * upstream * value_of(gg_row, factors[f]);
                    for (int32_t k = 0; k < order; k++) {
                        if (k != f && k != f2) {
                            term *= value_of(a_row, factors[k]);
                        }
                    }
                    second += term;
                }
                out_row[factors[f2]] += second;
            }
        }
    }
    if (grad_grad_output != nullptr) {
        grad_grad_output[row] = sum;
    }
}

// Rows per workgroup: as many as possible (fewer table reads per row) while
// the launch still has about a thousand workgroups and the tiles fit in LDS.
// Returns 0 when even R = 1 does not fit.
int pick_rows(size_t n_rows, size_t bytes_per_row) {
    int R = 64;
    while (R > 1 && (n_rows / R < 1024 || bytes_per_row * R > LDS_BUDGET)) {
        R >>= 1;
    }
    return bytes_per_row * R > LDS_BUDGET ? 0 : R;
}

} // namespace
} // namespace hpe
using namespace hpe;
} // namespace mops::amd

namespace mops::cuda {

template <typename scalar_t>
void homogeneous_polynomial_evaluation(MOPS_HPE_PARAMS(MOPS_CXX_FIRST, MOPS_CXX_NEXT)) {
    using namespace mops::amd;
    const char* operation = "cuda_homogeneous_polynomial_evaluation";
    checks::Validator validator(operation);
    checks::hpe(validator, output, A, C, indices_A);
    validate_gather_index(indices_A, A.shape[1], "indices_A", operation);

    const int32_t n_rows = narrow_i32(A.shape[0], "A.shape[0]");
    const int32_t nA = narrow_i32(A.shape[1], "A.shape[1]");
    const int32_t n_monomials = narrow_i32(indices_A.shape[0], "indices_A.shape[0]");
    const int32_t order = narrow_i32(indices_A.shape[1], "indices_A.shape[1]");
    if (n_rows == 0) {
        return;
    }
    hipStream_t stream = current_stream();
    const hpe_tiles::Shape shape{n_rows, nA, n_monomials, order};
    const auto kernels = thresholds::hpe_forward(n_rows, nA, static_cast<int64_t>(n_monomials) * order, sizeof(scalar_t));
    if (kernels == thresholds::HpeKernels::ROWS && hpe_rows::covers_forward(shape, sizeof(scalar_t))) {
        hpe_rows::forward<scalar_t>(output.data, A.data, C.data, indices_A.data, shape, stream);
        finish_call(operation);
        return;
    }
    const auto plan = hpe_tiles::plan_forward(shape, sizeof(scalar_t));
    const size_t bytes = hpe_tiles::forward_bytes(shape, plan, sizeof(scalar_t));
    if (plan.values > 0 && kernels != thresholds::HpeKernels::FEW && (bytes == 0 || scratch_ready(bytes))) {
        void* workspace = bytes > 0 ? scratch(bytes) : nullptr;
        auto launch = [&](int32_t* counters) {
            hpe_tiles::forward<scalar_t>(
                output.data, A.data, C.data, indices_A.data, shape, plan, workspace, counters, stream
            );
        };
        if (bytes > 0) {
            ScratchCounters counters;
            launch(counters.data());
        } else {
            launch(nullptr);
        }
        finish_call(operation);
        return;
    }
    constexpr int THREADS = 256;
    // per row: its A values plus one partial sum per group (G <= THREADS)
    int R = pick_rows(n_rows, (static_cast<size_t>(nA) + 1 + THREADS) * sizeof(scalar_t));
    if (R > 0) {
        size_t lds = ((static_cast<size_t>(nA) + 1) * R + THREADS) * sizeof(scalar_t);
        unsigned blocks = static_cast<unsigned>(ceil_div(static_cast<size_t>(n_rows), R));
        MainKernelTimer timer(stream);
#define MOPS_LAUNCH_ORDERED(ORDER)                                                                  \
    forward_ordered_kernel<scalar_t, ORDER><<<blocks, THREADS, lds, stream>>>(                     \
        output.data, A.data, C.data, indices_A.data, n_rows, nA, n_monomials, R                    \
    )
        switch (order) {
        case 0:
            MOPS_LAUNCH_ORDERED(0);
            break;
        case 1:
            MOPS_LAUNCH_ORDERED(1);
            break;
        case 2:
            MOPS_LAUNCH_ORDERED(2);
            break;
        case 3:
            MOPS_LAUNCH_ORDERED(3);
            break;
        case 4:
            MOPS_LAUNCH_ORDERED(4);
            break;
        case 5:
            MOPS_LAUNCH_ORDERED(5);
            break;
        case 6:
            MOPS_LAUNCH_ORDERED(6);
            break;
        default:
            forward_kernel<scalar_t><<<blocks, THREADS, lds, stream>>>(
                output.data, A.data, C.data, indices_A.data, n_rows, nA, n_monomials, order, R
            );
            break;
        }
#undef MOPS_LAUNCH_ORDERED
    } else {
        unsigned blocks = static_cast<unsigned>(ceil_div(static_cast<size_t>(n_rows), THREADS));
        forward_global_kernel<scalar_t><<<blocks, THREADS, 0, stream>>>(
            output.data, A.data, C.data, indices_A.data, n_rows, nA, n_monomials, order
        );
    }
    finish_call(operation);
}

template <typename scalar_t>
void homogeneous_polynomial_evaluation_vjp(MOPS_HPE_VJP_PARAMS(MOPS_CXX_FIRST, MOPS_CXX_NEXT)) {
    using namespace mops::amd;
    const char* operation = "cuda_homogeneous_polynomial_evaluation_vjp";
    checks::Validator validator(operation);
    checks::hpe_vjp(validator, grad_A, grad_output, A, C, indices_A);
    if (grad_A.data == nullptr) {
        return;
    }
    validate_gather_index(indices_A, A.shape[1], "indices_A", operation);

    const int32_t n_rows = narrow_i32(A.shape[0], "A.shape[0]");
    const int32_t nA = narrow_i32(A.shape[1], "A.shape[1]");
    const int32_t n_monomials = narrow_i32(indices_A.shape[0], "indices_A.shape[0]");
    const int32_t order = narrow_i32(indices_A.shape[1], "indices_A.shape[1]");
    if (n_rows == 0 || nA == 0) {
        return;
    }
    hipStream_t stream = current_stream();
    // accumulators of every feature for each of the 64 lanes that walk the monomials
    const size_t accumulator_bytes = (static_cast<size_t>(nA) + 1) * WAVE * sizeof(scalar_t);
    const hpe_tiles::Shape shape{n_rows, nA, n_monomials, order};
    const auto kernels = thresholds::hpe_vjp(n_rows, nA, static_cast<int64_t>(n_monomials) * order, sizeof(scalar_t));
    if (kernels == thresholds::HpeKernels::ROWS && hpe_rows::covers_vjp(shape, sizeof(scalar_t)) &&
        scratch_ready(hpe_tiles::table_bytes(shape, sizeof(scalar_t)))) {
        void* workspace = scratch(hpe_tiles::table_bytes(shape, sizeof(scalar_t)));
        hpe_rows::vjp<scalar_t>(
            grad_A.data, grad_output.data, A.data, C.data, indices_A.data, shape, workspace, stream
        );
        finish_call(operation);
        return;
    }
    const auto plan = hpe_tiles::plan_gradient(shape, sizeof(scalar_t), false);
    const size_t bytes = plan.values > 0 ? hpe_tiles::gradient_bytes(shape, plan, sizeof(scalar_t), false) : 0;
    if (plan.values > 0 && (kernels != thresholds::HpeKernels::FEW || accumulator_bytes > LDS_BUDGET) &&
        scratch_ready(bytes)) {
        void* workspace = scratch(bytes);
        hpe_tiles::vjp<scalar_t>(
            grad_A.data, grad_output.data, A.data, C.data, indices_A.data, shape, plan, workspace, stream
        );
        finish_call(operation);
        return;
    }
    // LDS holds R rows of A and the accumulators, whatever R is
    // Rows per workgroup: the fewest for which all workgroups are on the
    // device at once (256 CUs, as many workgroups per CU as the 160 KB of LDS
    // hold): a second round of workgroups costs more than rows twice as long
    // (c0: 17.8 us with 1000 workgroups of one row, 12.0 us with 500 of two, 17.2 us
    // with 250 of four).
    int R = 0;
    for (int rows = 1; rows <= 64 && R == 0; rows <<= 1) {
        const size_t lds = accumulator_bytes + (static_cast<size_t>(nA) + 1) * rows * sizeof(scalar_t);
        if (lds > LDS_BUDGET) {
            break;
        }
        const size_t resident = 256 * std::max<size_t>(1, (160 * 1024) / lds);
        if (ceil_div(static_cast<size_t>(n_rows), rows) <= resident || rows == 64) {
            R = rows;
        }
    }
    if (R == 0 && accumulator_bytes + (static_cast<size_t>(nA) + 1) * sizeof(scalar_t) <= LDS_BUDGET) {
        // the tiles of 64 rows do not fit: as many rows as do
        R = 1;
        while (accumulator_bytes + (static_cast<size_t>(nA) + 1) * (2 * R) * sizeof(scalar_t) <= LDS_BUDGET && R < 64) {
            R <<= 1;
        }
    }
    int32_t span = nA; // features whose accumulators one workgroup keeps
    if (R == 0 && (static_cast<size_t>(nA) + 1) * sizeof(scalar_t) <= LDS_BUDGET / 2) {
        // the accumulators of all features do not fit: one row per workgroup,
        // the features in ranges that do
        R = 1;
        span = static_cast<int32_t>(
            (LDS_BUDGET - (static_cast<size_t>(nA) + 1) * sizeof(scalar_t)) / (WAVE * sizeof(scalar_t)) - 1
        );
    }
    if (R > 0) {
        // (one row more of each than there are features: see vjp_ordered_kernel)
        size_t lds = (static_cast<size_t>(span) + 1) * WAVE * sizeof(scalar_t) +
                     (static_cast<size_t>(nA) + 1) * R * sizeof(scalar_t);
        int32_t log2_R = 0;
        while ((1 << log2_R) < R) {
            log2_R++;
        }
        const dim3 blocks(
            static_cast<unsigned>(ceil_div(static_cast<size_t>(n_rows), R)),
            static_cast<unsigned>(ceil_div(static_cast<size_t>(nA), span))
        );
        MainKernelTimer timer(stream);
#define MOPS_LAUNCH_ORDERED(ORDER)                                                                  \
    vjp_ordered_kernel<scalar_t, ORDER><<<blocks, ORDERED_VJP_THREADS, lds, stream>>>(             \
        grad_A.data, grad_output.data, A.data, C.data, indices_A.data, n_rows, nA, n_monomials,    \
        log2_R                                                                                     \
    )
        // (features in ranges: kernels of any order)
        switch (n_monomials > 0 && span == nA ? order : 0) {
        case 1:
            MOPS_LAUNCH_ORDERED(1);
            break;
        case 2:
            MOPS_LAUNCH_ORDERED(2);
            break;
        case 3:
            MOPS_LAUNCH_ORDERED(3);
            break;
        case 4:
            MOPS_LAUNCH_ORDERED(4);
            break;
        case 5:
            MOPS_LAUNCH_ORDERED(5);
            break;
        case 6:
            MOPS_LAUNCH_ORDERED(6);
            break;
        default:
            vjp_kernel<scalar_t><<<blocks, WAVE, lds, stream>>>(
                grad_A.data, grad_output.data, A.data, C.data, indices_A.data, n_rows, nA, n_monomials,
                order, R, span
            );
            break;
        }
#undef MOPS_LAUNCH_ORDERED
    } else {
        unsigned blocks = static_cast<unsigned>(ceil_div(static_cast<size_t>(n_rows), 256));
        vjp_global_kernel<scalar_t><<<blocks, 256, 0, stream>>>(
            grad_A.data, grad_output.data, A.data, C.data, indices_A.data, n_rows, nA, n_monomials, order
        );
    }
    finish_call(operation);
}

// Second order. The reference has it on the host only
// (mops/src/hpe/cpu.tpp:275-539; device: "Not implemented",
// mops/src/hpe/hpe.cu:402-413) and reads through a null grad_grad_A
// (cpu.tpp:367-388); here a cotangent that is not given counts as zero.
template <typename scalar_t>
void homogeneous_polynomial_evaluation_vjp_vjp(MOPS_HPE_VJP_VJP_PARAMS(MOPS_CXX_FIRST, MOPS_CXX_NEXT)) {
    using namespace mops::amd;
    const char* operation = "cuda_homogeneous_polynomial_evaluation_vjp_vjp";
    checks::Validator validator(operation);
    checks::hpe_vjp_vjp(validator, grad_grad_output, grad_A_2, grad_grad_A, grad_output, A, C, indices_A);
    if (grad_grad_output.data == nullptr && grad_A_2.data == nullptr) {
        return;
    }
    validate_gather_index(indices_A, A.shape[1], "indices_A", operation);

    const int32_t n_rows = narrow_i32(A.shape[0], "A.shape[0]");
    const int32_t nA = narrow_i32(A.shape[1], "A.shape[1]");
    const int32_t n_monomials = narrow_i32(indices_A.shape[0], "indices_A.shape[0]");
    const int32_t order = narrow_i32(indices_A.shape[1], "indices_A.shape[1]");
    if (n_rows == 0) {
        return;
    }
    hipStream_t stream = current_stream();
    if (grad_grad_A.data == nullptr || nA == 0) {
        if (grad_grad_output.data != nullptr) {
            fill_zero<scalar_t>(grad_grad_output.data, static_cast<size_t>(n_rows), stream);
        }
        if (grad_A_2.data != nullptr) {
            fill_zero<scalar_t>(grad_A_2.data, static_cast<size_t>(n_rows) * nA, stream);
        }
        finish_call(operation);
        return;
    }
    const size_t accumulator_bytes = (static_cast<size_t>(nA) + 1) * WAVE * sizeof(scalar_t);
    const hpe_tiles::Shape shape{n_rows, nA, n_monomials, order};
    const auto kernels = thresholds::hpe_vjp_vjp(n_rows, nA, static_cast<int64_t>(n_monomials) * order, sizeof(scalar_t));
    const auto plan = hpe_tiles::plan_gradient(shape, sizeof(scalar_t), true);
    const size_t bytes = plan.values > 0 ? hpe_tiles::gradient_bytes(shape, plan, sizeof(scalar_t), true) : 0;
    if (plan.values > 0 && (kernels != thresholds::HpeKernels::FEW || accumulator_bytes > LDS_BUDGET) &&
        scratch_ready(bytes)) {
        void* workspace = scratch(bytes);
        ScratchCounters counters;
        hpe_tiles::vjp_vjp<scalar_t>(
            grad_grad_output.data, grad_A_2.data, grad_grad_A.data, grad_output.data, A.data, C.data, indices_A.data,
            shape, plan, workspace, counters.data(), stream
        );
        finish_call(operation);
        return;
    }
    // order known at compile time: the tiles of vjp_ordered_kernel and one more of grad_grad_A;
    // rows per workgroup as there (the fewest for which all workgroups are on the device at once)
    if (order >= 1 && order <= 6 && n_monomials > 0) {
        auto ordered_lds = [&](int rows) {
            return accumulator_bytes + 2 * (static_cast<size_t>(nA) + 1) * rows * sizeof(scalar_t);
        };
        int log2_R = -1;
        for (int log2_rows = 0; log2_rows <= 6 && ordered_lds(1 << log2_rows) <= LDS_BUDGET; log2_rows++) {
            log2_R = log2_rows;
            const size_t resident = 256 * std::max<size_t>(1, (160 * 1024) / ordered_lds(1 << log2_rows));
            if (ceil_div(static_cast<size_t>(n_rows), size_t(1) << log2_rows) <= resident) {
                break;
            }
        }
        if (log2_R >= 0) {
            const unsigned blocks = static_cast<unsigned>(ceil_div(static_cast<size_t>(n_rows), size_t(1) << log2_R));
            const size_t lds = ordered_lds(1 << log2_R);
#define MOPS_LAUNCH_ORDERED(ORDER)                                                                  \
    vjp_vjp_ordered_kernel<scalar_t, ORDER><<<blocks, ORDERED_VJP_THREADS, lds, stream>>>(         \
        grad_grad_output.data, grad_A_2.data, grad_grad_A.data, grad_output.data, A.data, C.data,  \
        indices_A.data, n_rows, nA, n_monomials, log2_R                                            \
    )
            switch (order) {
            case 1:
                MOPS_LAUNCH_ORDERED(1);
                break;
            case 2:
                MOPS_LAUNCH_ORDERED(2);
                break;
            case 3:
                MOPS_LAUNCH_ORDERED(3);
                break;
            case 4:
                MOPS_LAUNCH_ORDERED(4);
                break;
            case 5:
                MOPS_LAUNCH_ORDERED(5);
                break;
            default:
                MOPS_LAUNCH_ORDERED(6);
                break;
            }
#undef MOPS_LAUNCH_ORDERED
            finish_call(operation);
            return;
        }
    }
    // LDS: 2 R rows (A and grad_grad_A), WAVE accumulator rows, WAVE partial sums
    const size_t fixed_bytes = (static_cast<size_t>(nA) + 1) * WAVE * sizeof(scalar_t);
    auto lds_for = [&](int rows) { return fixed_bytes + 2 * static_cast<size_t>(nA) * rows * sizeof(scalar_t); };
    int R = 64;
    while (R > 1 && (static_cast<size_t>(n_rows) / R < 1024 || lds_for(R) > LDS_BUDGET)) {
        R >>= 1;
    }
    if (lds_for(R) <= LDS_BUDGET) {
        const unsigned blocks = static_cast<unsigned>(ceil_div(static_cast<size_t>(n_rows), R));
        vjp_vjp_kernel<scalar_t><<<blocks, WAVE, lds_for(R), stream>>>(
            grad_grad_output.data, grad_A_2.data, grad_grad_A.data, grad_output.data, A.data, C.data,
            indices_A.data, n_rows, nA, n_monomials, order, R
        );
    } else {
        const unsigned blocks = static_cast<unsigned>(ceil_div(static_cast<size_t>(n_rows), 256));
        vjp_vjp_global_kernel<scalar_t><<<blocks, 256, 0, stream>>>(
            grad_grad_output.data, grad_A_2.data, grad_grad_A.data, grad_output.data, A.data, C.data,
            indices_A.data, n_rows, nA, n_monomials, order
        );
    }
    finish_call(operation);
}

MOPS_CXX_INSTANTIATE(homogeneous_polynomial_evaluation, MOPS_HPE_PARAMS)
MOPS_CXX_INSTANTIATE(homogeneous_polynomial_evaluation_vjp, MOPS_HPE_VJP_PARAMS)
MOPS_CXX_INSTANTIATE(homogeneous_polynomial_evaluation_vjp_vjp, MOPS_HPE_VJP_VJP_PARAMS)

} // namespace mops::cuda
