// The kernels of sap_rows.hpp for one element type (sap_rows_f32.hip,
// sap_rows_f64.hip: two files so that they compile beside each other).
//
//   O[i, o] = sum_{a, b} M[a, b, o] * (A[i, a] * B[i, b])
//
// A lane stands for row i, and M, the table made dense, is the same for all
// lanes: it comes in scalar registers, a row M[a, b, :] at a time, asked for one
// row ahead, and every multiply-add takes one scalar and two vector registers.
// Nothing is padded but the inner index (to an even number) and the columns (to
// a multiple of four), nothing goes between lanes, and both gradients come from
//
//   t = sum_o M[a, b, o] * gO[i, o],   grad_A[i, a] += t * B[i, b],   grad_B[i, b] += t * A[i, a]
//
// with ONE look at M, where the matrix cores (sap_mfma.hip) take a product of
// their own for each gradient. For double they multiply no faster than the
// vector units; in float twice as fast, of which padding to 16 and the second
// product leave nothing in the gradients.
//
// The lane keeps its values of the inner index (the one that pads better), its
// sums or its upstream gradients, and its gradients of the inner index in
// registers; those of the outer index are in LDS, a wavefront's own part of it,
// through which all rows also go in and out so that memory is read and written
// in order. No wavefront waits for another.
//
// M is made by a launch in front, a workgroup for each outer index and tile of
// columns (6 us of the calls below).
//
// A million rows of 13, 7 and 20 values, 900 entries, whole calls, matrix cores ->
// this, the same buffers every call: vjp 272 -> 133 us in double, 133 -> 83 in
// float; second order 606 -> 277 and 338 -> 178; forward pass in double 132 -> 113.
// Vector instructions occupy 0.77 (vjp, float), 0.55 (vjp, double) and 0.62
// (forward, double) of the SIMDs' clocks at 2.4 GHz in these kernels (98 rows of M,
// 20 multiply-adds each and 15 % of other work) and memory moves at 2.7 to 3.6
// TB/s; rows in and out alone would take 109 us (vjp, double) and 73 (forward) at
// the rate of a large copy.
#include "sap_rows.hpp"

#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "dispatch_thresholds.hpp"
#include "runtime.hpp"
#include "sasaw_table.hpp"

namespace mops::amd::sap_rows {
namespace {

using sasaw::BufferOf;
using sasaw::NOBODY;
using sasaw::unless;
using sasaw::wave_sync;

constexpr int WAVES = 4; // per workgroup
constexpr int THREADS = WAVES * WAVE;
constexpr int OUTER_AT_ONCE = 16; // values of the outer index a lane loads at a time

__host__ __device__ constexpr int32_t odd(int32_t n) { return n | 1; }

// ------------------------------------------------------------------- table --
constexpr int BUILD_THREADS = 1024;
static_assert(MAX_ENTRIES <= 32 * BUILD_THREADS, "a bit for each of a thread's entries");

/// dense[((tile * n_outer + outer) * inner_pad + inner) * columns + o - tile * columns]; one workgroup
/// per (outer, tile). LDS: a T and an integer for each of its inner_pad * columns cells.
template <typename T>
__global__ __launch_bounds__(BUILD_THREADS) void table_kernel(
    T* __restrict__ dense, const T* __restrict__ C, const int32_t* __restrict__ outer_of,
    const int32_t* __restrict__ inner_of, const int32_t* __restrict__ output_of, int32_t entries, int32_t n_outer,
    int32_t n_inner, int32_t inner_pad, int32_t n_out, int32_t columns
) {
    extern __shared__ __align__(16) char lds[];
    const int32_t cells = inner_pad * columns;
    T* cell = reinterpret_cast<T*>(lds);
    int32_t* owner = reinterpret_cast<int32_t*>(cell + cells);
    const int32_t outer = blockIdx.x % n_outer, first = blockIdx.x / n_outer * columns;
    const int32_t here = min(columns, n_out - first);
    for (int32_t i = threadIdx.x; i < cells; i += BUILD_THREADS) {
        cell[i] = T(0);
        owner[i] = NOBODY;
    }
    auto look = [&](int32_t k) {
        const int32_t a = outer_of[k], inner = inner_of[k], o = output_of[k] - first;
        return a == outer && in_bounds(inner, n_inner) && in_bounds(o, here) ? inner * columns + o : -1;
    };
    // (a thread's first entries stay in registers)
    const bool has[2] = {static_cast<int32_t>(threadIdx.x) < entries, static_cast<int32_t>(threadIdx.x) + BUILD_THREADS < entries};
    const int32_t safe[2] = {has[0] ? static_cast<int32_t>(threadIdx.x) : 0, has[1] ? static_cast<int32_t>(threadIdx.x) + BUILD_THREADS : 0};
    const T coefficient[2] = {C[safe[0]], C[safe[1]]};
    const int32_t looked[2] = {look(safe[0]), look(safe[1])};
    auto cell_of = [&](int32_t bit) {
        return bit == 0 ? looked[0] : bit == 1 ? looked[1] : look(threadIdx.x + bit * BUILD_THREADS);
    };
    // entries of one cell are added in ascending order: every round the smallest pending one of each
    uint32_t pending = (has[0] && looked[0] >= 0 ? 1u : 0u) | (has[1] && looked[1] >= 0 ? 2u : 0u);
    for (int32_t bit = 2; static_cast<int32_t>(threadIdx.x) + bit * BUILD_THREADS < entries; bit++) {
        pending |= cell_of(bit) >= 0 ? 1u << bit : 0u;
    }
    __syncthreads();
    do {
        for (uint32_t left = pending; left != 0; left &= left - 1) {
            const int32_t bit = __ffs(left) - 1;
            atomicMin(&owner[cell_of(bit)], static_cast<int32_t>(threadIdx.x + bit * BUILD_THREADS));
        }
        __syncthreads();
        uint32_t winners = 0;
        for (uint32_t left = pending; left != 0; left &= left - 1) {
            const int32_t bit = __ffs(left) - 1, k = static_cast<int32_t>(threadIdx.x) + bit * BUILD_THREADS, c = cell_of(bit);
            if (owner[c] == k) {
                cell[c] += bit == 0 ? coefficient[0] : bit == 1 ? coefficient[1] : C[k];
                winners |= 1u << bit;
            }
        }
        __syncthreads();
        for (uint32_t left = winners; left != 0; left &= left - 1) {
            owner[cell_of(__ffs(left) - 1)] = NOBODY;
        }
        pending &= ~winners;
    } while (__syncthreads_or(pending != 0));
    T* target = dense + static_cast<size_t>(blockIdx.x) * cells;
    for (int32_t i = threadIdx.x; i < cells; i += BUILD_THREADS) {
        target[i] = cell[i];
    }
}

// -------------------------------------------------------------------- rows --
/// `width` of the columns of 64 rows, which a wavefront takes as element i = 64 t + lane of [64][width].
struct Columns {
    int32_t width;
    uint32_t reciprocal; // ceil(2^20 / width): exact for the 64 width elements, width < 128, in 24-bit multiplications

    static __host__ Columns make(int32_t width) {
        return Columns{width, ((1u << 20) + static_cast<uint32_t>(width) - 1) / static_cast<uint32_t>(width)};
    }
    __device__ __forceinline__ uint32_t row(uint32_t i) const { return __umul24(i, reciprocal) >> 20; }
    /// In LDS, odd(width) elements per row, so that 64 lanes reading a row each meet 64 banks.
    __device__ __forceinline__ uint32_t staged(uint32_t i) const { return (width & 1) != 0 ? i : i + row(i); }
    /// In memory, n per row, from column `begin` on.
    __device__ __forceinline__ uint32_t place(uint32_t i, int32_t n, int32_t begin) const {
        return i + __umul24(row(i), static_cast<uint32_t>(n - width)) + static_cast<uint32_t>(begin);
    }
};

template <typename T> struct Arguments {
    T* output; // forward
    T* grad_outer;
    T* grad_inner;
    const T* grad_output;
    const T* outer;
    const T* inner;
    const T* outer2; // forward of two pairs
    const T* inner2;
    const T* dense;
    int32_t n_rows, n_outer, n_inner, n_out, tiles;
    int32_t touched; // bytes of the table to be touched
    Columns outer_columns, inner_columns, tile_columns, last_tile_columns;
    // a wavefront's LDS, in elements: all of it, where rows are staged, and where the outer index's
    // gradients are summed (the same place as its values if there is one tile only)
    int32_t area, staging, sums, second;
};

/// Row M[a, b, :] in scalar registers.
template <typename T, int OT> struct ScalarRow {
    typedef const __attribute__((address_space(4))) T* Uniform;
    T value[OT];

    __device__ __forceinline__ void ask(const T* from) {
        const Uniform row = (Uniform)from;
#pragma unroll
        for (int o = 0; o < OT; o++) {
            value[o] = row[o];
        }
    }
    __device__ __forceinline__ void arrived() {
#pragma unroll
        for (int o = 0; o < OT; o++) {
            asm volatile("" : "+s"(value[o]));
        }
    }
};

/// Makes the scalar cache, which two compute units share, hold a table of `bytes` bytes: a wavefront
/// that asked for one row after the other would wait for the L2 cache at each. Every wavefront of the
/// workgroup asks for its share of the lines, twelve on their way at a time (32 000 rows, where every
/// wavefront is the first: 25 -> 10.7 us).
__device__ __forceinline__ void touch(const void* table, int32_t bytes, int wave) {
    constexpr int32_t LINE = 64, AT_ONCE = 12;
    typedef const __attribute__((address_space(4))) int32_t* Uniform;
    const Uniform words = (Uniform)table;
    for (int32_t at = wave * LINE; at < bytes; at += WAVES * LINE * AT_ONCE) {
        int32_t word[AT_ONCE];
#pragma unroll
        for (int k = 0; k < AT_ONCE; k++) {
            word[k] = words[min(at + k * WAVES * LINE, bytes - 4) / 4];
        }
#pragma unroll
        for (int k = 0; k < AT_ONCE; k++) {
            asm volatile("" ::"s"(word[k]));
        }
    }
}

/// The 64 rows of a wavefront, a lane each.
template <typename T> struct Rows {
    int lane, wave;
    /// ... of which the compiler knows nothing: places in LDS are computed where they are used, and not
    /// kept in dozens of registers from one use to the next.
    __device__ __forceinline__ int fresh_lane() const {
        int fresh = lane;
        asm volatile("" : "+v"(fresh));
        return fresh;
    }
    int64_t first;
    int32_t count;

    /// Asks for columns begin .. of the rows of a tensor with n columns: element 64 t + lane of their
    /// [64][columns.width] in `to[t]`; beyond the rows and the columns, zero.
    template <int N>
    __device__ __forceinline__ void ask(T (&to)[N], const T* tensor, int32_t n, int32_t begin, Columns columns) const {
        const uint32_t lane = fresh_lane();
        const BufferOf<T> rows = buffer(tensor, n);
        if (columns.width == n) { // (uniform)
#pragma unroll
            for (int t = 0; t < N; t++) {
                to[t] = rows.load((t * WAVE + lane) * static_cast<uint32_t>(sizeof(T)), 0);
            }
        } else {
#pragma unroll
            for (int t = 0; t < N; t++) {
                to[t] = rows.load(columns.place(t * WAVE + lane, n, begin) * static_cast<uint32_t>(sizeof(T)), 0);
            }
        }
    }
    /// All columns, elements 64 (t0 + t) + lane.
    template <int N> __device__ __forceinline__ void ask_all(T (&to)[N], const T* tensor, int32_t n, int32_t t0) const {
        const uint32_t lane = fresh_lane();
        const BufferOf<T> rows = buffer(tensor, n);
#pragma unroll
        for (int t = 0; t < N; t++) {
            to[t] = rows.load(((t0 + t) * WAVE + lane) * static_cast<uint32_t>(sizeof(T)), 0);
        }
    }
    /// Puts what was asked for into an area of odd(columns.width) elements per row.
    template <int N>
    __device__ __forceinline__ void lay_out(T* area, const T (&asked)[N], Columns columns, int32_t t0 = 0) const {
        const uint32_t lane = fresh_lane();
#pragma unroll
        for (int t = 0; t < N; t++) {
            if (t0 + t < columns.width) { // (uniform)
                area[columns.staged((t0 + t) * WAVE + lane)] = asked[t];
            }
        }
    }
    /// What ask() brought, to the lanes whose rows it is; zero beyond the columns.
    template <int N>
    __device__ __forceinline__ void deal(T (&mine)[N], const T (&asked)[N], T* staging, Columns columns) const {
        lay_out(staging, asked, columns);
        wave_sync();
        const T* from = staging + fresh_lane() * odd(columns.width);
#pragma unroll
        for (int t = 0; t < N; t++) {
            mine[t] = from[t]; // (the area holds N columns and more)
        }
        if (columns.width < N) { // (uniform)
#pragma unroll
            for (int t = 0; t < N; t++) {
                mine[t] = t < columns.width ? mine[t] : T(0);
            }
        }
        wave_sync();
    }
    /// The other way: every lane's row to columns begin .. of the tensor.
    template <int N>
    __device__ __forceinline__ void
    put(T* tensor, int32_t n, int32_t begin, const T (&mine)[N], T* staging, Columns columns) const {
        T* to = staging + fresh_lane() * odd(columns.width);
#pragma unroll
        for (int t = 0; t < N; t++) {
            if (t < columns.width) { // (uniform)
                to[t] = mine[t];
            }
        }
        wave_sync();
        const uint32_t lane = fresh_lane();
        const BufferOf<T> rows = buffer(tensor, n);
#pragma unroll
        for (int t = 0; t < N; t++) {
            if (t < columns.width) { // (uniform)
                const uint32_t i = t * WAVE + lane;
                rows.store(
                    staging[columns.staged(i)],
                    (columns.width == n ? i : columns.place(i, n, begin)) * static_cast<uint32_t>(sizeof(T)), 0
                );
            }
        }
        wave_sync();
    }
    /// The area of all columns to the tensor.
    __device__ __forceinline__ void put_whole(T* tensor, const T* area, Columns columns) const {
        const uint32_t lane = fresh_lane();
        const BufferOf<T> rows = buffer(tensor, columns.width);
#pragma unroll 8
        for (int32_t t = 0; t < columns.width; t++) {
            const uint32_t i = t * WAVE + lane;
            rows.store(area[columns.staged(i)], i * static_cast<uint32_t>(sizeof(T)), 0);
        }
    }

    __device__ __forceinline__ BufferOf<T> buffer(const T* tensor, int32_t n) const {
        BufferOf<T> rows;
        rows.set(tensor + first * n, static_cast<uint32_t>(count * n) * sizeof(T));
        return rows;
    }
};

/// The kernel's arguments once more, for what comes after the loop (and rows_of_wave() also has
/// everything computed again): the compiler would keep what it knows from before in scalar registers, of
/// which the rows of M take all there are.
template <typename T> __device__ __forceinline__ const Arguments<T> arguments_again() {
    typedef const __attribute__((address_space(4))) Arguments<T>* Uniform;
    Uniform p = (Uniform)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const Arguments<T>*)p;
}

/// The wavefront's rows, false if it has none.
template <typename T> __device__ __forceinline__ bool rows_of_wave(Rows<T>& rows, int32_t n_rows) {
    uint32_t thread = threadIdx.x, block = blockIdx.x;
    asm volatile("" : "+v"(thread), "+s"(block));
    const int wave = __builtin_amdgcn_readfirstlane(thread / WAVE); // (uniform, and known to be)
    rows.wave = wave;
    rows.lane = thread & (WAVE - 1);
    rows.first = (static_cast<int64_t>(block) * WAVES + wave) * WAVE;
    rows.count = static_cast<int32_t>(min(static_cast<int64_t>(WAVE), n_rows - rows.first));
    return rows.count > 0;
}

/// The values of the outer index: the first ones are on their way.
template <typename T>
__device__ __forceinline__ void
outer_rows(const Rows<T>& rows, T* area, T (&asked)[OUTER_AT_ONCE], const T* tensor, Columns columns) {
    rows.lay_out(area, asked, columns);
    for (int32_t t0 = OUTER_AT_ONCE; t0 < columns.width; t0 += OUTER_AT_ONCE) {
        rows.ask_all(asked, tensor, columns.width, t0);
        rows.lay_out(area, asked, columns, t0);
    }
}

/// What bounds it: the multiply-adds; next the rows going in and out.
template <typename T, int NB, int OT, bool TWO>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(3))) void forward_kernel(const Arguments<T> p) {
    extern __shared__ __align__(16) char lds[];
    Rows<T> rows;
    if (!rows_of_wave(rows, p.n_rows)) {
        return;
    }
    T* area = reinterpret_cast<T*>(lds) + rows.wave * p.area;
    T* staging = area + p.staging;
    T asked_inner[NB], asked_outer[OUTER_AT_ONCE], inner[NB], inner2[TWO ? NB : 1];
    rows.ask_all(asked_inner, p.inner, p.n_inner, 0);
    rows.ask_all(asked_outer, p.outer, p.n_outer, 0);
    if constexpr (TWO) {
        T asked_inner2[NB], asked_outer2[OUTER_AT_ONCE];
        rows.ask_all(asked_inner2, p.inner2, p.n_inner, 0);
        rows.ask_all(asked_outer2, p.outer2, p.n_outer, 0);
        touch(p.dense, p.touched, rows.wave);
        rows.deal(inner, asked_inner, staging, p.inner_columns);
        rows.deal(inner2, asked_inner2, staging, p.inner_columns);
        outer_rows(rows, area, asked_outer, p.outer, p.outer_columns);
        outer_rows(rows, area + p.second, asked_outer2, p.outer2, p.outer_columns);
    } else {
        touch(p.dense, p.touched, rows.wave);
        rows.deal(inner, asked_inner, staging, p.inner_columns);
        outer_rows(rows, area, asked_outer, p.outer, p.outer_columns);
    }
    wave_sync();
    const int32_t pitch = odd(p.n_outer);
    const T* mine = area + rows.lane * pitch;
    const T* dense = p.dense;
    ScalarRow<T, OT> row[2];
    row[0].ask(dense);
    for (int32_t tile = 0; tile < p.tiles; tile++) {
        T sum[OT];
#pragma unroll
        for (int o = 0; o < OT; o++) {
            sum[o] = T(0);
        }
        T next = mine[0], next2 = TWO ? mine[p.second] : T(0);
        for (int32_t a = 0; a < p.n_outer; a++) {
            const T outer = next, outer2 = next2;
            next = mine[min(a + 1, p.n_outer - 1)];
            if constexpr (TWO) {
                next2 = mine[p.second + min(a + 1, p.n_outer - 1)];
            }
#pragma unroll
            for (int b = 0; b < NB; b++) {
                row[b & 1].arrived();
                dense += OT;
                row[~b & 1].ask(dense); // (after the last row of the table: one that is readable)
                __builtin_amdgcn_sched_barrier(0);
                T product = outer * inner[b];
                if constexpr (TWO) {
                    product += outer2 * inner2[b];
                }
#pragma unroll
                for (int o = 0; o < OT; o++) {
                    sum[o] += row[b & 1].value[o] * product;
                }
            }
        }
        const Arguments<T> q = arguments_again<T>();
        Rows<T> again;
        rows_of_wave(again, q.n_rows);
        wave_sync(); // (of a single tile, the sums take the place of the values)
        again.put(
            q.output, q.n_out, tile * OT, sum, reinterpret_cast<T*>(lds) + again.wave * q.area + q.staging,
            tile + 1 < q.tiles ? q.tile_columns : q.last_tile_columns
        );
    }
}

/// What bounds it: as above.
template <typename T, int NB, int OT>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(3))) void vjp_kernel(const Arguments<T> p) {
    extern __shared__ __align__(16) char lds[];
    Rows<T> rows;
    if (!rows_of_wave(rows, p.n_rows)) {
        return;
    }
    T* area = reinterpret_cast<T*>(lds) + rows.wave * p.area;
    T* staging = area + p.staging;
    T asked_inner[NB], asked_outer[OUTER_AT_ONCE], asked[OT], inner[NB], upstream[OT], grad_inner[NB];
    const Columns first = p.tiles > 1 ? p.tile_columns : p.last_tile_columns;
    rows.ask(asked, p.grad_output, p.n_out, 0, first);
    rows.ask_all(asked_inner, p.inner, p.n_inner, 0);
    rows.ask_all(asked_outer, p.outer, p.n_outer, 0);
    touch(p.dense, p.touched, rows.wave);
    rows.deal(upstream, asked, staging, first);
    rows.deal(inner, asked_inner, staging, p.inner_columns);
    outer_rows(rows, area, asked_outer, p.outer, p.outer_columns);
    wave_sync();
#pragma unroll
    for (int b = 0; b < NB; b++) {
        grad_inner[b] = T(0);
    }
    const int32_t pitch = odd(p.n_outer);
    T* mine = area + rows.lane * pitch;
    T* sums = mine + p.sums;
    const T* dense = p.dense;
    ScalarRow<T, OT> row[2];
    row[0].ask(dense);
    for (int32_t tile = 0; tile < p.tiles; tile++) {
        if (tile > 0) {
            const Columns columns = tile + 1 < p.tiles ? p.tile_columns : p.last_tile_columns;
            rows.ask(asked, p.grad_output, p.n_out, tile * OT, columns);
            rows.deal(upstream, asked, staging, columns);
        }
        T next = mine[0];
        for (int32_t a = 0; a < p.n_outer; a++) {
            const T outer = next;
            next = mine[min(a + 1, p.n_outer - 1)];
            T grad_outer = tile > 0 ? sums[a] : T(0);
#pragma unroll
            for (int b = 0; b < NB; b++) {
                row[b & 1].arrived();
                dense += OT;
                row[~b & 1].ask(dense);
                __builtin_amdgcn_sched_barrier(0);
                T even = row[b & 1].value[0] * upstream[0], uneven = row[b & 1].value[1] * upstream[1];
#pragma unroll
                for (int o = 2; o < OT; o += 2) {
                    even += row[b & 1].value[o] * upstream[o];
                    uneven += row[b & 1].value[o + 1] * upstream[o + 1];
                }
                const T t = even + uneven;
                grad_outer += t * inner[b];
                grad_inner[b] += t * outer;
            }
            sums[a] = grad_outer;
        }
    }
    wave_sync();
    const Arguments<T> q = arguments_again<T>();
    Rows<T> again;
    rows_of_wave(again, q.n_rows);
    T* area_again = reinterpret_cast<T*>(lds) + again.wave * q.area;
    if (q.grad_outer != nullptr) {
        again.put_whole(q.grad_outer, area_again + q.sums, q.outer_columns);
        wave_sync();
    }
    if (q.grad_inner != nullptr) {
        again.put(q.grad_inner, q.n_inner, 0, grad_inner, area_again + q.staging, q.inner_columns);
    }
}

// -------------------------------------------------------------------- host --
/// body(inner values, columns)
template <typename T, typename Body> void with_sizes(int32_t inner, int32_t columns, Body&& body) {
    auto with_inner = [&](auto nb) {
        switch (columns) {
        case 4:
            return body(nb, std::integral_constant<int, 4>{});
        case 8:
            return body(nb, std::integral_constant<int, 8>{});
        case 12:
            return body(nb, std::integral_constant<int, 12>{});
        case 16:
            return body(nb, std::integral_constant<int, 16>{});
        case 20:
            return body(nb, std::integral_constant<int, 20>{});
        default:
            if constexpr (sizeof(T) == 4) {
                switch (columns) {
                case 24:
                    return body(nb, std::integral_constant<int, 24>{});
                case 28:
                    return body(nb, std::integral_constant<int, 28>{});
                default:
                    return body(nb, std::integral_constant<int, 32>{});
                }
            }
        }
    };
    switch (inner) {
    case 4:
        return with_inner(std::integral_constant<int, 4>{});
    case 6:
        return with_inner(std::integral_constant<int, 6>{});
    case 8:
        return with_inner(std::integral_constant<int, 8>{});
    case 10:
        return with_inner(std::integral_constant<int, 10>{});
    case 12:
        return with_inner(std::integral_constant<int, 12>{});
    case 14:
        return with_inner(std::integral_constant<int, 14>{});
    default:
        return with_inner(std::integral_constant<int, 16>{});
    }
}

template <typename Kernel> void allow_lds(Kernel kernel, size_t bytes) {
    if (bytes > 64 * 1024) {
        MOPS_HIP_CHECK(hipFuncSetAttribute(
            reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)
        ));
    }
}

/// The sizes, and M.
template <typename T>
Arguments<T> prepare(const Table& table, const Shape& s, bool A_inside, int32_t inner_pad, const Tiles& tiles, hipStream_t stream) {
    Arguments<T> p{};
    p.n_rows = s.n_rows;
    p.n_outer = A_inside ? s.nB : s.nA;
    p.n_inner = A_inside ? s.nA : s.nB;
    p.n_out = s.nO;
    p.tiles = tiles.count;
    p.outer_columns = Columns::make(p.n_outer);
    p.inner_columns = Columns::make(p.n_inner);
    p.tile_columns = Columns::make(tiles.columns);
    p.last_tile_columns = Columns::make(s.nO - (tiles.count - 1) * tiles.columns);
    const size_t cells = static_cast<size_t>(inner_pad) * tiles.columns;
    const size_t blocks = static_cast<size_t>(tiles.count) * p.n_outer;
    T* dense = static_cast<T*>(scratch(scratch_bytes(s, sizeof(T))));
    p.dense = dense;
    p.touched = static_cast<int32_t>(blocks * cells * sizeof(T));
    const size_t lds = cells * (sizeof(T) + sizeof(int32_t));
    table_kernel<T><<<static_cast<unsigned>(blocks), BUILD_THREADS, lds, stream>>>(
        dense, static_cast<const T*>(table.C), A_inside ? table.indices_B : table.indices_A,
        A_inside ? table.indices_A : table.indices_B, table.indices_output, s.K, p.n_outer, p.n_inner, inner_pad, s.nO,
        tiles.columns
    );
    return p;
}

} // namespace

template <typename T>
void forward(
    T* output, const T* A, const T* B, const T* A2, const T* B2, const Table& table, const Shape& s, hipStream_t stream
) {
    const bool A_inside = inner_is_A(s), two = A2 != nullptr;
    const Tiles tiles = tiles_of(s.nO, sizeof(T));
    const int32_t inner_pad = padded(A_inside ? s.nA : s.nB);
    Arguments<T> p = prepare<T>(table, s, A_inside, inner_pad, tiles, stream);
    p.output = output;
    p.outer = A_inside ? B : A;
    p.inner = A_inside ? A : B;
    p.outer2 = A_inside ? B2 : A2;
    p.inner2 = A_inside ? A2 : B2;
    const int32_t values = WAVE * odd(p.n_outer), staged = WAVE * std::max(odd(tiles.columns), odd(inner_pad));
    p.second = two ? values : 0;
    p.staging = tiles.count == 1 ? 0 : (two ? 2 : 1) * values;
    p.area = std::max((two ? 2 : 1) * values, p.staging + staged);
    MainKernelTimer timer(stream);
    with_sizes<T>(inner_pad, tiles.columns, [&](auto nb, auto columns) {
        constexpr int NB = decltype(nb)::value, OT = decltype(columns)::value;
        const size_t lds = static_cast<size_t>(WAVES) * p.area * sizeof(T);
        const unsigned blocks = static_cast<unsigned>(ceil_div(static_cast<size_t>(s.n_rows), THREADS));
        auto launch = [&](auto kernel) {
            allow_lds(kernel, lds);
            kernel<<<blocks, THREADS, lds, stream>>>(p);
        };
        if (two) {
            launch(forward_kernel<T, NB, OT, true>);
        } else {
            launch(forward_kernel<T, NB, OT, false>);
        }
    });
    MOPS_HIP_CHECK(hipGetLastError());
}

template <typename T>
void vjp(
    T* grad_A, T* grad_B, const T* grad_output, const T* A, const T* B, const Table& table, const Shape& s,
    hipStream_t stream
) {
    const bool A_inside = inner_is_A(s);
    const Tiles tiles = tiles_of(s.nO, sizeof(T));
    const int32_t inner_pad = padded(A_inside ? s.nA : s.nB);
    Arguments<T> p = prepare<T>(table, s, A_inside, inner_pad, tiles, stream);
    p.grad_output = grad_output;
    p.outer = A_inside ? B : A;
    p.inner = A_inside ? A : B;
    p.grad_outer = A_inside ? grad_B : grad_A;
    p.grad_inner = A_inside ? grad_A : grad_B;
    const int32_t values = WAVE * odd(p.n_outer), staged = WAVE * std::max(odd(tiles.columns), odd(inner_pad));
    p.sums = tiles.count == 1 ? 0 : values;
    p.staging = tiles.count == 1 ? 0 : 2 * values;
    p.area = std::max(values, p.staging + staged);
    MainKernelTimer timer(stream);
    with_sizes<T>(inner_pad, tiles.columns, [&](auto nb, auto columns) {
        constexpr int NB = decltype(nb)::value, OT = decltype(columns)::value;
        const size_t lds = static_cast<size_t>(WAVES) * p.area * sizeof(T);
        const unsigned blocks = static_cast<unsigned>(ceil_div(static_cast<size_t>(s.n_rows), THREADS));
        auto kernel = vjp_kernel<T, NB, OT>;
        allow_lds(kernel, lds);
        kernel<<<blocks, THREADS, lds, stream>>>(p);
    });
    MOPS_HIP_CHECK(hipGetLastError());
}

} // namespace mops::amd::sap_rows
