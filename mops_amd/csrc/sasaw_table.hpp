// What the kernels of SASAW share (sasaw_segments.hip, sasaw_columns.hip): the
// coupling table made dense in LDS, in the layouts of matrix operands, and
// tensors as buffers.
#ifndef MOPS_AMD_SASAW_TABLE_HPP
#define MOPS_AMD_SASAW_TABLE_HPP

#include <cstdint>

#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "dispatch_thresholds.hpp"

namespace mops::amd::sasaw {

constexpr int MAX_INDEX = thresholds::SASAW_INDEX_VALUES; // values of a component index
constexpr int ENTRIES_PER_LANE = 4;    // table entries a lane of the building wavefront handles at a time
constexpr int MAX_TABLE = 1 << 16;     // entries (more: the general kernels)

// ---------------------------------------------------------------------------
// the dense table in LDS
//
// For a contraction whose gathered blocks have `n_red` rows (m2 in the forward
// pass) and whose result has `n_out` rows (m3 in the forward pass):
//
//   table[(r * n_red + c) * 64 + 16 * q + o] = D[o, c, m1(q, r)]
//
// i.e. for every register r of an accumulator tile and every block row c, the
// left operand (lane = o + 16 q) of the product with that register. m1(q, r)
// is the component of A that row `Mfma<T>::row(16 q, r)` of the accumulators
// stands for.

/// Component of A in accumulator row `row` (0..15); >= nA: none. Rows whose
/// register number is beyond `registers` = ceil(nA / 4) hold nothing, so that
/// the second product needs `registers` steps per block row and not four.
template <typename T> __host__ __device__ __forceinline__ int32_t component_of_row(int row, int32_t registers) {
    if constexpr (sizeof(T) == 4) {
        const int q = row >> 2, r = row & 3; // row = 4 q + r
        return r < registers ? registers * q + r : 4 * MAX_INDEX;
    } else {
        return row; // row = 4 r + q
    }
}

/// (q, r) of component m1: inverse of the above.
template <typename T> __device__ __forceinline__ void place_of_component(int32_t m1, int32_t registers, int& q, int& r) {
    if constexpr (sizeof(T) == 4) {
        q = m1 / registers;
        r = m1 - q * registers;
    } else {
        r = m1 >> 2;
        q = m1 & 3;
    }
}

/// The layouts the dense table is needed in. All are "what one lane of a
/// wavefront holds as an operand of one matrix instruction, instruction after
/// instruction", so that reading it is one conflict-free LDS access.
enum class Layout : int32_t {
    // result = D * sums (contract_kernel, and grad_W): see above
    RESULT,
    // grad_A: right operand of (grad_output of a node)^T * D[:, m2, :], per
    // block row m2 and step s3 over the rows of the result:
    //   table[((m2 * steps3 + s3) * 64 + 16 * k + m1] = D[4 * s3 + k, m2, m1]
    ALPHA,
    // grad_B: left operand of D' * (grad_output of a node), whose rows are
    // pairs (component of A, block row) in the order the accumulators of the
    // next product want them: pair p = s * bucket + m2 (s = m1 / 4) lies in
    // tile p / 4, register p % 4, of the lanes q = m1 % 4:
    //   table[((p / 4) * steps3 + s3) * 64 + 16 * k + row(q, p % 4)] = D[4 * s3 + k, m2, m1]
    BETA
};

struct Table {
    const int32_t* PA;   // [N]
    const int32_t* Pred; // [N] index of the block row that is summed over (forward: PW2)
    const int32_t* Pout; // [N] index of the row of the result (forward: PO2)
    int32_t N, nA, n_red, n_out;
    int32_t registers; // ceil(nA / 4)
    Layout layout;
    int32_t bucket; // BETA: accumulator tiles of the kernel (>= n_red)
    // The part of the coupling table this launch works with: components m1_begin .. m1_begin + nA
    // of A, block rows red_begin .. red_begin + n_red, rows out_begin .. out_begin + n_out of the
    // result (all zero and the whole ranges for shapes that one launch covers). RESULT only:
    // n_out may exceed 16; the rows of the result then come in blocks of 16.
    int32_t m1_begin, red_begin, out_begin;

    __host__ __device__ int32_t steps3() const { return (n_out + 3) / 4; }
    __host__ __device__ int32_t slots() const {
        switch (layout) {
        case Layout::ALPHA:
            return n_red * steps3() * WAVE;
        case Layout::BETA:
            return (registers * bucket + 3) / 4 * steps3() * WAVE;
        default:
            return out_blocks() * registers * n_red * WAVE;
        }
    }
    __host__ __device__ int32_t out_blocks() const { return (n_out + 15) / 16; }
};

/// Where D[o, c, m1] goes (all three inside their ranges).
template <typename T> __device__ __forceinline__ int32_t slot_in(const Table& t, int32_t m1, int32_t c, int32_t o) {
    switch (t.layout) {
    case Layout::ALPHA:
        return (c * t.steps3() + (o >> 2)) * WAVE + 16 * (o & 3) + m1;
    case Layout::BETA: {
        const int32_t pair = (m1 >> 2) * t.bucket + c;
        const int q = m1 & 3, r = pair & 3;
        const int row = sizeof(T) == 4 ? 4 * q + r : 4 * r + q;
        return ((pair >> 2) * t.steps3() + (o >> 2)) * WAVE + 16 * (o & 3) + row;
    }
    default: {
        int q, r;
        place_of_component<T>(m1, t.registers, q, r);
        return (((o >> 4) * t.registers + r) * t.n_red + c) * WAVE + 16 * q + (o & 15);
    }
    }
}

constexpr int32_t NOBODY = 0x7fffffff;

/// Orders LDS traffic between the lanes of one wavefront.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/// Table entries `first` + lane + 64 k (k < ENTRIES_PER_LANE) of one lane, as
/// loaded (asked for at the start of a kernel, looked at when the table is built).
template <typename T> struct MyEntries {
    int32_t m1[ENTRIES_PER_LANE], c[ENTRIES_PER_LANE], o[ENTRIES_PER_LANE];
    T coefficient[ENTRIES_PER_LANE];
};

template <typename T>
__device__ __forceinline__ void load_entries(
    MyEntries<T>& mine, const T* __restrict__ C, const Table& t, int32_t first, int lane
) {
#pragma unroll
    for (int k = 0; k < ENTRIES_PER_LANE; k++) {
        const int32_t n = first + lane + k * WAVE;
        const int32_t safe = n < t.N ? n : 0;
        mine.m1[k] = t.PA[safe];
        mine.c[k] = t.Pred[safe];
        mine.o[k] = t.Pout[safe];
        mine.coefficient[k] = C[safe];
    }
}

/// The dense table, built by ONE wavefront (all 64 lanes call this): nothing
/// in it waits for another wavefront, so the others are free to ask for their
/// first rows meanwhile; they meet the builder at one barrier afterwards.
/// `owner` is an array of slots() integers. `mine`: load_entries(.., first = 0, ..).
template <typename T>
__device__ __forceinline__ void build_table(
    T* __restrict__ table, int32_t* __restrict__ owner, MyEntries<T>& mine, const T* __restrict__ C, const Table& t,
    int lane
) {
    const int32_t n_slots = t.slots();
    for (int32_t s = lane; s < n_slots; s += WAVE) {
        table[s] = T(0);
        owner[s] = NOBODY;
    }
    wave_sync();
    for (int32_t first = 0; first < t.N; first += WAVE * ENTRIES_PER_LANE) {
        if (first > 0) {
            load_entries<T>(mine, C, t, first, lane);
        }
        // where each entry goes (-1: nowhere; an entry outside the tensors is dropped)
        int32_t slot[ENTRIES_PER_LANE];
        uint32_t pending = 0;
#pragma unroll
        for (int k = 0; k < ENTRIES_PER_LANE; k++) {
            const int32_t n = first + lane + k * WAVE;
            const int32_t m1 = mine.m1[k] - t.m1_begin, c = mine.c[k] - t.red_begin, o = mine.o[k] - t.out_begin;
            const bool inside = n < t.N && in_bounds(m1, t.nA) && in_bounds(c, t.n_red) && in_bounds(o, t.n_out);
            slot[k] = inside ? slot_in<T>(t, m1, c, o) : -1;
            pending |= inside ? 1u << k : 0u;
        }
        // Every round the smallest pending entry of each slot is added to it: the
        // entries of one slot in ascending order. (LDS operations of one
        // wavefront happen in program order.)
        while (__ballot(pending != 0) != 0) {
#pragma unroll
            for (int k = 0; k < ENTRIES_PER_LANE; k++) {
                if ((pending >> k) & 1u) {
                    atomicMin(&owner[slot[k]], first + lane + k * WAVE);
                }
            }
            wave_sync();
            uint32_t winners = 0;
#pragma unroll
            for (int k = 0; k < ENTRIES_PER_LANE; k++) {
                if (((pending >> k) & 1u) && owner[slot[k]] == first + lane + k * WAVE) {
                    winners |= 1u << k;
                    table[slot[k]] += mine.coefficient[k];
                }
            }
            wave_sync();
#pragma unroll
            for (int k = 0; k < ENTRIES_PER_LANE; k++) {
                if ((winners >> k) & 1u) {
                    owner[slot[k]] = NOBODY;
                }
            }
            pending &= ~winners;
            wave_sync();
        }
    }
}

/// A tensor as a buffer: loads are a uniform descriptor, a 32-bit byte offset
/// per lane and a uniform byte offset (the hardware adds the three), and an
/// offset beyond the tensor reads as zero without touching memory. That is one
/// address register per lane for all the rows of a block, and lanes without an
/// edge need no row that exists: they ask beyond the end.
template <typename T> struct BufferOf {
    __amdgpu_buffer_rsrc_t descriptor;

    __device__ __forceinline__ void set(const T* base, uint32_t bytes) {
        // (word 3: 32-bit data format, as the other libraries of this platform set it for gfx9)
        descriptor = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, static_cast<int>(bytes), 0x00020000);
    }
    __device__ __forceinline__ T load(uint32_t lane_bytes, uint32_t uniform_bytes) const {
        if constexpr (sizeof(T) == 4) {
            return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(descriptor, lane_bytes, uniform_bytes, 0));
        } else {
            return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(descriptor, lane_bytes, uniform_bytes, 0));
        }
    }
    /// (nothing is stored at an offset beyond the tensor)
    __device__ __forceinline__ void store(T value, uint32_t lane_bytes, uint32_t uniform_bytes) const {
        if constexpr (sizeof(T) == 4) {
            __builtin_amdgcn_raw_buffer_store_b32(
                __builtin_bit_cast(uint32_t, value), descriptor, lane_bytes, uniform_bytes, 0
            );
        } else {
            typedef uint32_t Two __attribute__((ext_vector_type(2)));
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(Two, value), descriptor, lane_bytes, uniform_bytes, 0);
        }
    }
};
constexpr uint32_t BEYOND = 0xffffffffu; // a byte offset no tensor reaches (the host sends larger ones elsewhere)

/// All ones unless `wanted`: OR-ed into a byte offset it makes the load read
/// zero. (Arithmetic instead of a choice between an offset and a constant: the
/// compiler turns such a choice in front of a load into two branches.)
__device__ __forceinline__ uint32_t unless(bool wanted) { return static_cast<uint32_t>(wanted) - 1u; }

} // namespace mops::amd::sasaw

#endif
