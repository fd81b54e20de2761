// SASAW with a lane per feature column, for gfx950.
//
//   Z_i[m1, m2, l] = sum over edges e of i of  A[e, m1] * (B[e, l] * W[PW1[e], m2, l])
//   O[i, m3, l]    = sum_{m1, m2} D[m3, m2, m1] * Z_i[m1, m2, l]
//
// (D: the coupling table made dense, see sasaw_segments.hip.) A lane stands for
// a column l and keeps sums of Z_i[:, :, l] of a node in registers; an edge is
// then a multiply-add per sum, whose operands are the edge's row of A, the same
// for all lanes and therefore in scalar registers, and the lane's own elements
// of B and of the rows of W. No lane works on padding but where the columns or
// the block rows do not fill a wavefront, nothing is exchanged between lanes
// until the node's edges are done, and the addresses of an edge are scalar
// arithmetic. The f32 matrix cores do the same products at the same rate per
// useful operation only if all 16 rows of an instruction are useful (9 of 16 at
// l <= 2), and the f64 ones at half of it.
//
// The 64 lanes are (part, column): tiles of 16, 32 or 64 columns, and 4, 2 or 1
// parts that share the block rows m2. What bounds these kernels is the
// multiply-adds and the latency of the gathered rows of W; several edges are on
// their way while one is worked on. O = D Z then goes through LDS and the
// matrix cores, a few components of A at a time.
//
// grad_A and grad_B of an edge need
//
//   U[m1, l]     = sum_m2 G_i[m1, m2, l] * W[PW1[e], m2, l],   G_i = D^T grad_output_i
//   grad_B[e, l] = sum_m1 A[e, m1] U[m1, l],   grad_A[e, m1] = sum_l B[e, l] U[m1, l]
//
// with G_i[:, :, l] of the receiver in the registers of the lane: both come from
// the same multiply-adds and ONE look at the rows of W; the sum over the columns
// is taken across lanes (DPP and permlane swaps). Of up to 9 components a lane has
// all block rows, and two or four edges of a node are worked on side by side: no
// sums across parts, no rows that fill the last part, and the sums over the columns
// of several edges for the instructions of one (an edge of 9 components and 32
// columns takes 72 vector instructions instead of 108 in float; 1 000 000 edges,
// grad_A and grad_B, f32 / f64: 245 -> 215 / 458 -> 410 us, 16 columns 197 -> 122;
// 60 000 edges 25.4 -> 22.2 / 36.2 -> 30.6). grad_W is the sum of the
// forward pass over the edges of a sender, with the roles of W and grad_output,
// m2 and m3 exchanged.
//
// Whole calls against one per-node sum on the matrix cores each, 9 components, 32
// columns, the same buffers every call, f32 / f64, us: 1 000 000 edges, forward 315
// -> 200 / 391 -> 370, vjp 1184 -> 447 / 1397 -> 812; 60 000 edges, 20.2 -> 20.2 /
// 29.2 -> 25.1 and 58.5 -> 46 / 99 -> 59.5; 128 columns there, vjp 247 -> 108 / 360
// -> 201; 600 edges, 12.6 -> 7.4 / 14.0 -> 8.2 and 25.1 -> 11.0 / 31.7 -> 12.1. At a
// million edges 1.3 GB (float; 2.6 in double) come through the memory side of L2 in
// the forward pass, rows of W in no order for the most part, at 6.4 (7.1) TB/s: the
// same loads with nothing done to what they bring take 175 of the 200 us, and with
// twice as many on their way the time is the same.
//
// Every sum has one fixed order; no atomics on floating point.
#include "sasaw_columns.hpp"

#include <algorithm>
#include <type_traits>
#include <utility>

#include "device_common.hpp"
#include "mfma.hpp"
#include "runtime.hpp"
#include "sasaw_table.hpp"
#include "sender_buckets.hpp"
#include "sender_shares.hpp"

namespace mops::amd::sasaw_columns {
namespace {

using namespace mops::amd::sasaw;

constexpr int THREADS = 256;
constexpr int WAVES = THREADS / WAVE;

/// The sums of a lane for N components of A and N block rows: all components
/// times M2 block rows, a PARTS-th of them: part, part + PARTS, ... (so that the
/// parts together load consecutive rows). With EDGES > 1 the lanes work on that many
/// edges side by side instead, and every lane has all rows.
template <int N_, int COLUMNS_, int EDGES_ = 1> struct Sums {
    static constexpr int N = N_, COLUMNS = COLUMNS_, EDGES = EDGES_;
    static constexpr int PARTS = WAVE / COLUMNS / EDGES;
    static_assert(EDGES == 1 || PARTS == 1, "parts or edges");
    static constexpr int M2 = (N + PARTS - 1) / PARTS;
    static constexpr bool EXACT = PARTS * M2 == N;
    static constexpr int MC = N == 4 ? 4 : N == 9 ? 3 : 2; // components of A that go through LDS at a time
    static constexpr int CHUNKS = (N + MC - 1) / MC;
    static constexpr int VALUES = MC * M2;       // of a lane at a time
    static constexpr int PAIRS = PARTS * VALUES; // of a column at a time
    static constexpr int STEPS = (PAIRS + 3) / 4, TILES = (PAIRS + 15) / 16;
};

/// A tile of COLUMNS columns: an LDS row a little longer, so that four rows of
/// 16 columns, which a matrix instruction takes at a time, lie on different banks.
template <int COLUMNS> constexpr int pitch() { return COLUMNS == 16 ? 16 : COLUMNS + 16; }

// ------------------------------------------------------------------- table --
/// The dense table in LDS as operands of matrix instructions. Component m1 and
/// block row m2 are pair (m2 % PARTS) * VALUES + (m1 % MC) * M2 + m2 / PARTS of chunk m1 / MC.
///   SPREAD false (D as left operand of D * Z), step ks of 4 pairs:
///     table[(chunk * STEPS + ks) * 64 + 16 * (pair % 4) + o]
///   SPREAD (D^T as left operand of D^T * grad_output), tile zt of 16 pairs, step s3 of 4 rows:
///     table[((chunk * TILES + zt) * 4 + s3) * 64 + 16 * (o % 4) + pair % 16]
struct Dense {
    const int32_t* PA;   // [N]
    const int32_t* Pred; // [N] block row
    const int32_t* Pout; // [N] row of the result
    int32_t entries, n_out;
};
template <typename S, bool SPREAD> constexpr int table_slots() {
    return S::CHUNKS * (SPREAD ? S::TILES * 4 : S::STEPS) * WAVE;
}
template <typename S, bool SPREAD> __device__ __forceinline__ int32_t slot_of(int32_t m1, int32_t m2, int32_t o) {
    const int32_t chunk = m1 / S::MC;
    const int32_t pair = m2 % S::PARTS * S::VALUES + m1 % S::MC * S::M2 + m2 / S::PARTS;
    return SPREAD ? ((chunk * S::TILES + (pair >> 4)) * 4 + (o >> 2)) * WAVE + 16 * (o & 3) + (pair & 15)
                  : (chunk * S::STEPS + (pair >> 2)) * WAVE + 16 * (pair & 3) + o;
}

/// Called by all threads of a workgroup, which is in step afterwards. The
/// entries of one slot are added in ascending order: every round the smallest
/// pending one of each slot (`owner`: as many integers as the table has slots).
/// `meanwhile()`: what there is to do while the first entries are on their way.
template <typename T, typename S, bool SPREAD, typename Meanwhile>
__device__ __forceinline__ void build(
    T* __restrict__ table, int32_t* __restrict__ owner, const T* __restrict__ C, const Dense& t, Meanwhile&& meanwhile
) {
    constexpr int ENTRIES = 4; // of a thread at a time
    for (int32_t s = threadIdx.x; s < table_slots<S, SPREAD>(); s += THREADS) {
        table[s] = T(0);
        owner[s] = NOBODY;
    }
    for (int32_t first = 0; first < t.entries; first += THREADS * ENTRIES) {
        int32_t m1[ENTRIES], c[ENTRIES], o[ENTRIES], slot[ENTRIES];
        T coefficient[ENTRIES];
#pragma unroll
        for (int k = 0; k < ENTRIES; k++) {
            const int32_t safe = min(static_cast<int32_t>(first + threadIdx.x + k * THREADS), t.entries - 1);
            m1[k] = t.PA[safe];
            c[k] = t.Pred[safe];
            o[k] = t.Pout[safe];
            coefficient[k] = C[safe];
        }
        if (first == 0) {
            meanwhile();
        }
        uint32_t pending = 0;
#pragma unroll
        for (int k = 0; k < ENTRIES; k++) {
            const int32_t n = first + threadIdx.x + k * THREADS;
            const bool inside =
                n < t.entries && in_bounds(m1[k], S::N) && in_bounds(c[k], S::N) && in_bounds(o[k], t.n_out);
            slot[k] = slot_of<S, SPREAD>(m1[k], c[k], o[k]);
            pending |= inside ? 1u << k : 0u;
        }
        __syncthreads();
        do {
#pragma unroll
            for (int k = 0; k < ENTRIES; k++) {
                if (pending >> k & 1) {
                    atomicMin(&owner[slot[k]], static_cast<int32_t>(first + threadIdx.x + k * THREADS));
                }
            }
            __syncthreads();
            uint32_t winners = 0;
#pragma unroll
            for (int k = 0; k < ENTRIES; k++) {
                if ((pending >> k & 1) && owner[slot[k]] == static_cast<int32_t>(first + threadIdx.x + k * THREADS)) {
                    winners |= 1u << k;
                    table[slot[k]] += coefficient[k];
                }
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < ENTRIES; k++) {
                if (winners >> k & 1) {
                    owner[slot[k]] = NOBODY;
                }
            }
            pending &= ~winners;
        } while (__syncthreads_or(static_cast<int>(pending)));
    }
    __syncthreads();
}

// ---------------------------------------------------------------- wavefront --
template <typename T> __device__ __forceinline__ void swap_rows(T& x, T& y) { // odd rows of 16 lanes of x, even ones of y
    uint32_t a[sizeof(T) / 4], b[sizeof(T) / 4];
    __builtin_memcpy(a, &x, sizeof(T));
    __builtin_memcpy(b, &y, sizeof(T));
#pragma unroll
    for (size_t i = 0; i < sizeof(T) / 4; i++) {
        const auto swapped = __builtin_amdgcn_permlane16_swap(a[i], b[i], false, false);
        a[i] = swapped[0];
        b[i] = swapped[1];
    }
    __builtin_memcpy(&x, a, sizeof(T));
    __builtin_memcpy(&y, b, sizeof(T));
}
template <typename T> __device__ __forceinline__ void swap_halves(T& x, T& y) { // upper half of x, lower half of y
    uint32_t a[sizeof(T) / 4], b[sizeof(T) / 4];
    __builtin_memcpy(a, &x, sizeof(T));
    __builtin_memcpy(b, &y, sizeof(T));
#pragma unroll
    for (size_t i = 0; i < sizeof(T) / 4; i++) {
        const auto swapped = __builtin_amdgcn_permlane32_swap(a[i], b[i], false, false);
        a[i] = swapped[0];
        b[i] = swapped[1];
    }
    __builtin_memcpy(&x, a, sizeof(T));
    __builtin_memcpy(&y, b, sizeof(T));
}
/// Lanes 0-31: the two halves of x added up; lanes 32-63: those of y.
template <typename T> __device__ __forceinline__ T sum_halves(T x, T y) {
    swap_halves(x, y);
    return x + y;
}
/// Rows 0 and 2 of 16 lanes: row pairs of x added up; rows 1 and 3: those of y.
template <typename T> __device__ __forceinline__ T sum_rows(T x, T y) {
    swap_rows(x, y);
    return x + y;
}
/// The sum over the 16 lanes of a row, in all of them.
template <int CONTROL, typename T> __device__ __forceinline__ T rotated(T x) {
    uint32_t a[sizeof(T) / 4];
    __builtin_memcpy(a, &x, sizeof(T));
#pragma unroll
    for (size_t i = 0; i < sizeof(T) / 4; i++) {
        a[i] = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(a[i]), CONTROL, 0xf, 0xf, true));
    }
    __builtin_memcpy(&x, a, sizeof(T));
    return x;
}
template <typename T> __device__ __forceinline__ T sum_of_row(T x) {
    x += rotated<0x128>(x); // row_ror:8, 4, 2, 1
    x += rotated<0x124>(x);
    x += rotated<0x122>(x);
    x += rotated<0x121>(x);
    return x;
}

/// body(integral_constant 0), body(integral_constant 1), ..
template <typename Body, int... I>
__device__ __forceinline__ void unrolled(std::integer_sequence<int, I...>, Body&& body) {
    (body(std::integral_constant<int, I>{}), ...);
}

/// Sums over the COLUMNS lanes of an edge of COUNT values at once: every level adds up pairs of lanes, and where
/// there are two values, one half of the pairs goes on with the one and the other half with the other (three
/// instructions for two values; the sum of each on its own in all lanes is two, but then all the levels
/// after it are twice the work). The lane whose bits, in the order of the levels, are those of i ends with value i.
template <int COLUMNS, int COUNT, int LEVEL = COLUMNS == 32 ? 0 : 1, typename T, int SIZE>
__device__ __forceinline__ T folded(T (&value)[SIZE], const bool (&bit)[4]) {
    if constexpr (LEVEL == 5) {
        static_assert(COUNT == 1, "as many levels as it takes");
        return value[0];
    } else {
        // pairs of rows, mirrors of a row and of its halves, lanes two and one apart
        constexpr int CONTROL = LEVEL == 1 ? 0x140 : LEVEL == 2 ? 0x141 : LEVEL == 3 ? 0x4e : 0xb1;
#pragma unroll
        for (int k = 0; k < (COUNT + 1) / 2; k++) {
            const bool two = 2 * k + 1 < COUNT;
            const T x = value[2 * k], y = value[two ? 2 * k + 1 : 2 * k];
            if constexpr (LEVEL == 0) {
                value[k] = sum_rows(x, y);
            } else {
                const bool mine = bit[LEVEL - 1];
                value[k] = two ? (mine ? y : x) + rotated<CONTROL>(mine ? x : y) : x + rotated<CONTROL>(x);
            }
        }
        return folded<COLUMNS, (COUNT + 1) / 2, LEVEL + 1>(value, bit);
    }
}

/// First position of the sorted index (n entries) whose value is not below `value`.
__device__ __forceinline__ int32_t lower_bound(const int32_t* __restrict__ index, int32_t n, int32_t value, int lane) {
    int32_t low = 0, high = n;
    while (high - low > WAVE) {
        const int32_t step = (high - low + WAVE - 1) / WAVE;
        const int32_t probe = low + (lane + 1) * step - 1;
        const bool below = probe < high && index[min(probe, n - 1)] < value;
        const int32_t passed = __popcll(__ballot(below));
        low += passed * step;
        high = min(high, low + step);
    }
    const bool below = low + lane < high && index[min(low + lane, n - 1)] < value;
    return low + __popcll(__ballot(below));
}

/// The first positions whose values are not below `value` and not below `value` + 1: both searches at once, so
/// that they wait together (few nodes, forward, f32: 7.6 -> 7.4 us at 600 edges, 16.3 -> 15.8 at 8000 of 30).
__device__ __forceinline__ void bounds_of(
    const int32_t* __restrict__ index, int32_t n, int32_t value, int lane, int32_t& first, int32_t& end
) {
    int32_t low[2] = {0, 0}, high[2] = {n, n};
    bool more;
    do {
        int32_t step[2], probe[2], found[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            step[k] = max((high[k] - low[k] + WAVE - 1) / WAVE, 1);
            probe[k] = low[k] + (lane + 1) * step[k] - 1;
            found[k] = index[min(probe[k], n - 1)];
        }
        more = false;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int32_t passed = __popcll(__ballot(probe[k] < high[k] && found[k] < value + k));
            low[k] += passed * step[k];
            high[k] = min(high[k], low[k] + step[k]);
            more = more || step[k] > 1;
        }
    } while (more); // (after a step of one place, `low` is the answer)
    first = low[0];
    end = low[1];
}

template <typename T> struct Walk {
    const T* A;    // [n_edges][N]
    const T* B;    // [n_edges][L]
    const T* rows; // [n_blocks][N][L]  (forward: W)
    const T* C;    // [entries]
    int32_t n_edges, n_blocks, L;
    int32_t column_tiles;
    int32_t ranges; // of nodes or edges, a wavefront each (and tile)
    const int32_t* sorted; // [n_edges] node of every position, non-decreasing
    const int32_t* gather; // [n_edges] block of `rows` of every edge
    Dense table;
};

/// The next 64 positions of the sorted index, one per lane, asked for while the
/// ones before are worked on.
template <typename T> struct Window {
    int32_t receiver, source;
    bool inside;

    __device__ __forceinline__ Window(const Walk<T>& p, int32_t at, int32_t lane) {
        const int32_t position = min(at + lane, p.n_edges - 1);
        inside = at + lane < p.n_edges;
        receiver = p.sorted[position];
        source = p.gather[position];
    }
    /// How many of them, from the first on, name `node`.
    __device__ __forceinline__ int32_t edges_of(int32_t node) const {
        const unsigned long long others = __ballot(!inside || receiver != node);
        return others == 0 ? WAVE : __ffsll(others) - 1;
    }
};

/// A lane's place, and the rows of an edge it works on.
template <typename T, typename S> struct Columns {
    static constexpr int N = S::N, COLUMNS = S::COLUMNS, EDGES = S::EDGES, M2 = S::M2;
    /// Edges whose operands are on their way while one is worked on (of each of the EDGES).
    static constexpr int AHEAD = (M2 + 1) * sizeof(T) <= 32 ? 4 : 2;

    const Walk<T>& p;
    int lane, c, part, slot;
    int32_t column;
    bool column_inside;
    uint32_t column_bytes;
    uint32_t row_at[M2]; // byte offset of the lane's element of its rows in a block (a row there is not: the last)
    uint32_t row_bytes, block_bytes;
    BufferOf<T> B;

    /// What a lane loads for an edge. The row of A is the same for all lanes: a scalar load.
    struct Operands {
        T b;
        T w[M2];
        T more; // (edge_kernel)
    };
    typedef const __attribute__((address_space(4))) T* Uniform;

    __device__ __forceinline__ explicit Columns(const Walk<T>& walk) : p(walk) {
        lane = threadIdx.x & (WAVE - 1);
        c = lane & (COLUMNS - 1);
        part = EDGES == 1 ? lane / COLUMNS : 0;
        slot = EDGES == 1 ? 0 : lane / COLUMNS;
        row_bytes = static_cast<uint32_t>(p.L) * sizeof(T);
        block_bytes = N * row_bytes;
        B.set(p.B, static_cast<uint32_t>(p.n_edges) * row_bytes);
    }

    __device__ __forceinline__ void set_tile(int32_t tile) {
        column = tile * COLUMNS + c;
        column_inside = column < p.L;
        column_bytes = static_cast<uint32_t>(min(column, p.L - 1)) * sizeof(T);
#pragma unroll
        for (int m = 0; m < M2; m++) {
            row_at[m] = column_bytes + static_cast<uint32_t>(min(m * S::PARTS + part, N - 1)) * row_bytes;
        }
    }

    /// Whether the lane's row m exists (the others repeat the last one).
    __device__ __forceinline__ bool has_row(int m) const { return S::EXACT || m * S::PARTS + part < N; }

    /// Asks for the operands of an edge (edge and source are uniform). The rows of a source outside
    /// the tensor are those of a tensor of no bytes, which reads as zeros.
    __device__ __forceinline__ void load(Operands& to, int32_t edge, int32_t source) const {
        to.b = B.load(column_bytes, static_cast<uint32_t>(edge) * row_bytes);
        const bool exists = in_bounds(source, p.n_blocks);
        const uint32_t block = exists ? static_cast<uint32_t>(source) * block_bytes : 0;
        BufferOf<T> rows;
        rows.set(p.rows, exists ? static_cast<uint32_t>(p.n_blocks) * block_bytes : 0);
#pragma unroll
        for (int m = 0; m < M2; m++) {
            to.w[m] = rows.load(row_at[m], block);
        }
    }
    __device__ __forceinline__ void load_row_of_A(T (&to)[N], int32_t edge) const {
        const Uniform row = (Uniform)(p.A + static_cast<size_t>(static_cast<uint32_t>(edge)) * N);
#pragma unroll
        for (int i = 0; i < N; i++) {
            to[i] = row[i];
        }
    }

    /// `each(row of A, operands, k)` for the edges k < n <= 64 of a list: edge k is `edge_of(k)`, lane k
    /// holds its source (of one outside the tensor, everything counts as zero). `ask(operands, k)`:
    /// what else `each` wants loaded for an edge.
    ///
    /// What makes the operands of AHEAD edges be on their way: no branch between the asking and the
    /// waiting (the compiler counts the loads of both ways and takes the smaller number), the order of
    /// the asking kept, stores without a branch around them (they count as well), and rows of A
    /// asked for only when the ones before have arrived (scalar loads come back in any order, so that a
    /// wait is for all of them).
    ///
    /// A_BATCH: the rows of A asked for at once, while as many are worked on.
    /// `meanwhile()`: what there is to do while the first operands are on their way.
    template <int A_BATCH, typename EdgeOf, typename Ask, typename Meanwhile, typename Each>
    __device__ __forceinline__ void
    over(int32_t sources, int32_t n, EdgeOf&& edge_of, Ask&& ask_more, Meanwhile&& meanwhile, Each&& each) const {
        Operands ring[AHEAD];
        auto ask = [&](Operands& to, int32_t k) {
            k = min(k, n - 1);
            load(to, edge_of(k), __builtin_amdgcn_readlane(sources, k));
            ask_more(to, k);
            __builtin_amdgcn_sched_barrier(0);
        };
        T a[2][A_BATCH][N];
        auto ask_rows = [&](T (&to)[A_BATCH][N], int32_t k) {
#pragma unroll
            for (int r = 0; r < A_BATCH; r++) {
                load_row_of_A(to[r], edge_of(min(k + r, n - 1)));
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        ask_rows(a[0], 0);
#pragma unroll
        for (int d = 0; d < AHEAD; d++) {
            ask(ring[d], d);
        }
        meanwhile();
        auto step = [&](int d, int32_t k) {
            T(&rows)[A_BATCH][N] = a[d / A_BATCH & 1];
            if (d % A_BATCH == 0) {
#pragma unroll
                for (int r = 0; r < A_BATCH; r++) {
                    arrived(rows[r]);
                }
                ask_rows(a[~(d / A_BATCH) & 1], k + A_BATCH);
            }
            each(rows[d % A_BATCH], ring[d % AHEAD], k);
        };
        constexpr int STEPS = AHEAD > 2 * A_BATCH ? AHEAD : 2 * A_BATCH;
        int32_t first = 0;
        for (; first + STEPS <= n; first += STEPS) {
#pragma unroll
            for (int d = 0; d < STEPS; d++) {
                step(d, first + d);
                ask(ring[d % AHEAD], first + d + AHEAD);
            }
        }
#pragma unroll
        for (int d = 0; d < STEPS - 1; d++) {
            if (first + d >= n) { // (uniform; the two ways do not meet before the end)
                return;
            }
            step(d, first + d);
            if (d + AHEAD < STEPS - 1) {
                ask(ring[d % AHEAD], first + d + AHEAD);
            }
        }
    }

    /// EDGES > 1: `each(operands, first, valid)` for the edges at positions `first` to first + EDGES, one per slot,
    /// of the n <= 64 from `begin` on, whose sources the lanes hold; `valid`: whether the lane's is one of them.
    /// (Loads are counted as in `over`. An edge's row of A comes as an element per lane of every row of 16 lanes,
    /// from where the multiply-adds take it.)
    struct Side {
        T a, b, more;
        T w[M2];
    };
    template <typename Ask, typename Meanwhile, typename Each>
    __device__ __forceinline__ void side_by_side(
        const BufferOf<T>& A, const BufferOf<T>& rows, int32_t sources, int32_t begin, int32_t n, Ask&& ask_more,
        Meanwhile&& meanwhile, Each&& each
    ) const {
        const uint32_t a_at = static_cast<uint32_t>(slot * N + min(lane & 15, N - 1)) * static_cast<uint32_t>(sizeof(T));
        const uint32_t b_at = static_cast<uint32_t>(slot) * row_bytes + column_bytes;
        // (a source outside the tensor: an offset beyond it, also with what is added)
        const uint32_t block = static_cast<uint32_t>(sources) * block_bytes | unless(in_bounds(sources, p.n_blocks));
        const int32_t groups = (n + EDGES - 1) / EDGES;
        Side ring[AHEAD];
        auto ask = [&](Side& to, int32_t group) {
            const int32_t k = min(group, groups - 1) * EDGES;
            const uint32_t edge = static_cast<uint32_t>(begin + k);
            const uint32_t of_edge = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute((k + slot) << 2, static_cast<int>(block)));
            const uint32_t at = __builtin_elementwise_add_sat(of_edge, column_bytes);
#pragma unroll
            for (int m = 0; m < M2; m++) {
                to.w[m] = rows.load(at, m * row_bytes);
            }
            to.b = B.load(b_at, edge * row_bytes);
            to.a = A.load(a_at, edge * static_cast<uint32_t>(N * sizeof(T)));
            ask_more(to, edge);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int d = 0; d < AHEAD; d++) {
            ask(ring[d], d);
        }
        meanwhile();
        auto step = [&](int d, int32_t group) {
            each(ring[d], static_cast<uint32_t>(begin + group * EDGES), group * EDGES + slot < n);
        };
        int32_t first = 0;
        for (; first + AHEAD <= groups; first += AHEAD) {
#pragma unroll
            for (int d = 0; d < AHEAD; d++) {
                step(d, first + d);
                ask(ring[d], first + d + AHEAD);
            }
        }
#pragma unroll
        for (int d = 0; d < AHEAD - 1; d++) {
            if (first + d >= groups) { // (uniform)
                return;
            }
            step(d, first + d);
        }
    }

    /// Waits for a row of A.
    static __device__ __forceinline__ void arrived(T (&a)[N]) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            asm volatile("" : "+s"(a[i]));
        }
    }
};

// -------------------------------------------------------------- contraction --
template <typename T> struct ContractArgs {
    Walk<T> walk;
    T* result; // [n_blocks][n_out][L]
    const int32_t* senders; // [n_edges] LISTS == LOOKED_FOR
    EdgesBySender ordered;  // LISTS == ORDERED
    Shares shares;          // LISTS == BUCKETS
    SharePlan plan;
};

/// Where the edges of a node are: next to each other in the (sorted) index, in a list of all edges by node, in a
/// bucket that the workgroup fetches first, or anywhere in a short index that the workgroup looks through.
enum Lists { SEGMENTS, ORDERED, BUCKETS, LOOKED_FOR };

/// Rows of A in scalar registers at once, where they fit without others being moved out of the way:
/// 1 000 000 edges, 32 columns, 4 components, f32 / f64, 94.9 -> 92.7 / 198 -> 188 us, sums over
/// senders 180 -> 170 / 273 -> 264; 9 in double 386 -> 371; 9 in float is slower by it.
template <typename T, int N> constexpr int contract_rows_of_A() {
    return N == 4 ? 4 : N == 9 && sizeof(T) == 8 ? 2 : 1;
}
/// Wavefronts per SIMD.
template <typename T, int N, int COLUMNS> constexpr int contract_waves() {
    constexpr int REGISTERS = (N * Sums<N, COLUMNS>::M2 + 34) * static_cast<int>(sizeof(T)) / 4;
    return REGISTERS <= 90 ? 4 : REGISTERS <= 130 ? 3 : 2;
}
template <typename T, int N, int COLUMNS> constexpr size_t contract_lds() {
    using S = Sums<N, COLUMNS>;
    return table_slots<S, false>() * sizeof(T) +
           std::max(table_slots<S, false>() * sizeof(int32_t), WAVES * S::STEPS * 4 * pitch<COLUMNS>() * sizeof(T));
}
/// The same with a bucket's edges between the table and the stages, and what fetching them takes where the stages are.
__host__ __device__ constexpr size_t kept_of_bucket(int32_t per_bucket) {
    return (static_cast<size_t>(bucket_lds(per_bucket)) + 3) / 4 * 4 * sizeof(int32_t);
}
template <typename T, int N, int COLUMNS> constexpr size_t contract_lds(int32_t per_bucket) {
    constexpr size_t table = table_slots<Sums<N, COLUMNS>, false>() * sizeof(T);
    return table + kept_of_bucket(per_bucket) +
           std::max(contract_lds<T, N, COLUMNS>() - table, gather_lds<THREADS>(per_bucket) * sizeof(int32_t));
}

/// SHARED: a workgroup has one node, whose edges its wavefronts share; else every wavefront has a range of
/// nodes. Bound by the rows it gathers (many edges), by the chain of a node's edges (few). With no more
/// nodes than workgroups at a time, a node's 30 edges are a chain of eight: 600 edges, 9 components, 32
/// columns, f32 / f64, 11.3 -> 7.4 / 12.0 -> 8.2 us, 5000 edges 10.6 -> 8.8 / 11.7 -> 10.6. Beyond, the
/// same share-out of a range of nodes costs a table and a wait more for each share: 60 000 edges 19.3 -> 20.5.
/// (Ranges of equal edges instead of equal nodes: within 3 % either way from 100 000 to 1 000 000 edges.)
template <typename T, int N, int COLUMNS, Lists LISTS, bool SHARED>
__device__ __forceinline__ void contract(const ContractArgs<T>& args, char* lds, const int32_t block) {
    using M = Mfma<T>;
    using S = Sums<N, COLUMNS>;
    constexpr int M2 = S::M2, PITCH = pitch<COLUMNS>(), STAGE = S::STEPS * 4 * PITCH;
    constexpr int ROWS_OF_A = contract_rows_of_A<T, N>();
    const Walk<T>& p = args.walk;
    T* table = reinterpret_cast<T*>(lds);
    T* stages = table + table_slots<S, false>();
    int32_t* const kept = reinterpret_cast<int32_t*>(stages);
    if constexpr (LISTS == BUCKETS) {
        stages = reinterpret_cast<T*>(reinterpret_cast<char*>(stages) + kept_of_bucket(args.plan.per_bucket));
    }
    int32_t* const owner = reinterpret_cast<int32_t*>(stages); // (while the table is built)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE); // (uniform, and known to be)
    T* stage = stages + wave * STAGE;

    Columns<T, S> columns_of(p);
    const int lane = columns_of.lane;
    BucketEdges bucket{};
    // SHARED: (range, tile) by workgroup; of a bucket, its nodes and their tiles as wavefronts are done with the ones
    // before; else (range, tile) by wavefront.
    const int32_t unit = SHARED ? block : LISTS == BUCKETS ? block * p.column_tiles : block * WAVES + wave;
    const int32_t range = unit / p.column_tiles;
    int32_t tile = unit % p.column_tiles;
    if constexpr (LISTS == BUCKETS) {
        BucketFetch fetch(args.shares, args.plan, range);
        build<T, S, false>(table, owner, p.C, p.table, [&] { fetch.ask(); });
        bucket = gather_bucket<THREADS>(kept, owner, fetch, args.shares, args.plan, range, tile);
    } else {
        build<T, S, false>(table, owner, p.C, p.table, [] {});
    }
    for (int32_t k = lane; k < STAGE; k += WAVE) {
        stage[k] = T(0); // (rows of a step that stand for no pair stay zero)
    }
    wave_sync();
    if (range >= p.ranges) {
        return;
    }
    const int32_t node0 = LISTS == BUCKETS ? args.plan.first_of(range)
                                           : static_cast<int32_t>(static_cast<int64_t>(p.n_blocks) * range / p.ranges);
    const int32_t node1 = LISTS == BUCKETS
                              ? args.plan.first_of(range + 1)
                              : static_cast<int32_t>(static_cast<int64_t>(p.n_blocks) * (range + 1) / p.ranges);
    columns_of.set_tile(tile);

    T z[N * M2];
    auto add = [&](const T (&a)[N], const auto& operands, int32_t) {
        T bw[M2];
#pragma unroll
        for (int m = 0; m < M2; m++) {
            bw[m] = operands.b * operands.w[m];
        }
#pragma unroll
        for (int i = 0; i < N; i++) {
#pragma unroll
            for (int m = 0; m < M2; m++) {
                z[i * M2 + m] += a[i] * bw[m];
            }
        }
    };

    auto nothing = [](auto&, int32_t) {};
    auto not_now = [] {};

    // O = D Z, MC components of A at a time through LDS
    const int row16 = lane >> 4;
    T* mine = stage + columns_of.part * S::VALUES * PITCH + columns_of.c;
    const T* right = stage + row16 * PITCH + (lane & 15);
    auto finish = [&](int32_t node) {
        typename M::Acc acc[COLUMNS / 16];
#pragma unroll
        for (int t = 0; t < COLUMNS / 16; t++) {
            acc[t] = M::zero();
        }
#pragma unroll
        for (int chunk = 0; chunk < S::CHUNKS; chunk++) {
#pragma unroll
            for (int k = 0; k < S::VALUES; k++) { // pair k of the lane's part
                if (chunk * S::VALUES + k < N * M2) {
                    const T sum = z[chunk * S::VALUES + k];
                    mine[k * PITCH] = columns_of.has_row(k % M2) ? sum : T(0);
                }
            }
            wave_sync();
#pragma unroll
            for (int ks = 0; ks < S::STEPS; ks++) {
                const T left = table[(chunk * S::STEPS + ks) * WAVE + lane];
#pragma unroll
                for (int t = 0; t < COLUMNS / 16; t++) {
                    acc[t] = M::mma(left, right[4 * ks * PITCH + 16 * t], acc[t]);
                }
            }
            wave_sync();
        }
        if constexpr (SHARED) { // the sum over the wavefronts, in their order, by the first
            constexpr int VALUES = 4 * (COLUMNS / 16);
            static_assert(VALUES * WAVE <= STAGE, "a result fits a stage");
            if (wave > 0) {
#pragma unroll
                for (int k = 0; k < VALUES; k++) {
                    stage[k * WAVE + lane] = acc[k / 4][k % 4];
                }
            }
            __syncthreads();
            if (wave > 0) {
                return;
            }
#pragma unroll
            for (int other = 1; other < WAVES; other++) {
#pragma unroll
                for (int k = 0; k < VALUES; k++) {
                    acc[k / 4][k % 4] += stages[other * STAGE + k * WAVE + lane];
                }
            }
        }
        T* target = args.result + static_cast<size_t>(node) * p.table.n_out * p.L;
#pragma unroll
        for (int t = 0; t < COLUMNS / 16; t++) {
            const int32_t column = tile * COLUMNS + 16 * t + (lane & 15);
            if (column < p.L) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int row = M::row(lane, r);
                    if (row < p.table.n_out) {
                        target[static_cast<size_t>(row) * p.L + column] = acc[t][r];
                    }
                }
            }
        }
    };
    auto clear = [&] {
#pragma unroll
        for (int k = 0; k < N * M2; k++) {
            z[k] = T(0);
        }
    };

    if constexpr (LISTS == LOOKED_FOR) {
        clear();
        const int32_t share = (p.n_edges + WAVES - 1) / WAVES, begin = min(wave * share, p.n_edges);
        edges_of_sender<4>(
            args.senders, p.n_edges, begin, min(begin + share, p.n_edges), node0, lane,
            [&](int32_t edge, int32_t n) {
                columns_of.template over<ROWS_OF_A>(
                    p.gather[edge], n, [&](int32_t k) { return __builtin_amdgcn_readlane(edge, k); }, nothing, not_now, add
                );
            }
        );
        finish(node0);
    } else {
        // Positions of the index or of a list from `at` on, one per lane, asked for while the ones before are worked
        // on: what is there (a node, or an edge), and the block of the edge.
        struct Positions {
            int32_t name, source;
            bool inside;
        };
        auto positions = [&](int32_t at) {
            Positions here;
            const int32_t last = LISTS == BUCKETS ? max(bucket.n, 1) : p.n_edges;
            const int32_t position = min(at + lane, last - 1);
            here.inside = at + lane < last;
            if constexpr (LISTS == SEGMENTS) {
                here.name = p.sorted[position];
                here.source = p.gather[position];
            } else {
                if constexpr (LISTS == ORDERED) {
                    here.name = args.ordered.edge[position];
                } else {
                    here.name = bucket.fits ? bucket.list[position] : bucket.in_memory[position];
                }
                here.source = p.gather[here.name];
            }
            return here;
        };
        auto begin_of = [&](int32_t node) { // (of a list)
            return LISTS == ORDERED ? args.ordered.offsets[node]
                                    : __builtin_amdgcn_readfirstlane(bucket.offsets[node - node0]);
        };
        // the sum over n edges at `at`, and what lies at `next`
        auto add_up = [&](Positions& here, int32_t at, int32_t n, int32_t next) {
            const Positions there = positions(next);
            if (n > 0) {
                columns_of.template over<ROWS_OF_A>(
                    here.source, n,
                    [&](int32_t k) { return LISTS == SEGMENTS ? at + k : __builtin_amdgcn_readlane(here.name, k); },
                    nothing, not_now, add
                );
            }
            here = there;
        };
        if constexpr (SHARED) { // the wavefront's quarter of the node's edges
            int32_t first, last;
            if constexpr (LISTS == SEGMENTS) {
                bounds_of(p.sorted, p.n_edges, node0, lane, first, last);
            } else {
                first = begin_of(node0);
                last = begin_of(node0 + 1);
            }
            int32_t at = first + static_cast<int32_t>(static_cast<int64_t>(last - first) * wave / WAVES), n;
            const int32_t to = first + static_cast<int32_t>(static_cast<int64_t>(last - first) * (wave + 1) / WAVES);
            Positions here = positions(at);
            clear();
            do {
                n = min(WAVE, to - at);
                add_up(here, at, n, at + n);
                at += n;
            } while (n == WAVE);
            finish(node0);
        } else if constexpr (LISTS == BUCKETS) {
            // One tile: whichever node is next when a wavefront is done with one. Several: up to four of them (step) of
            // a node at the same time, which share the lines that gathered rows lie on; each wavefront has every
            // WAVES / step-th node then. Three tiles leave a wavefront over: it has the last quarter of the nodes,
            // a tile of them after the other (of fewer than four nodes: as with one tile). 16 components, f32, W alone, 300 000
            // edges of 10 000 nodes, 40 columns: whichever is next 235 us, the third tile by itself 237, this 213;
            // 9 components, 32 columns, 1 000 000 edges: a quarter of the nodes each 250, whichever is next 241.
            struct Unit {
                int32_t node, tile, step;
            };
            const int32_t last_quarter = node1 - (node1 - node0) / 4;
            auto alone = [&](const Unit& unit) { return unit.step == 3 && wave == 3; };
            const bool any = p.column_tiles == 1 || (p.column_tiles == 3 && node1 - node0 < 4);
            auto nth = [&](int32_t k) { return Unit{node0 + k / p.column_tiles, k % p.column_tiles, 1}; };
            auto begin_tiles = [&](int32_t tile) { // (the first unit of this or of a later group of tiles)
                for (;;) {
                    const int32_t left = p.column_tiles - tile, step = min(left, 4);
                    const bool of_last = step == 3 && wave == 3;
                    const Unit unit{
                        of_last ? last_quarter : node0 + wave / max(step, 1), of_last ? tile : tile + wave % max(step, 1), step};
                    if (left <= 0 || unit.node < node1) {
                        return unit;
                    }
                    tile += step;
                }
            };
            auto exists = [&](const Unit& unit) { return unit.node < node1 && unit.tile < p.column_tiles; };
            Unit unit = any ? nth(wave) : begin_tiles(0);
            int32_t at = exists(unit) ? begin_of(unit.node) : 0, n;
            Positions here = positions(at);
            while (exists(unit)) {
                Unit next = unit;
                if (any) {
                    int32_t taken = 0;
                    if (lane == 0) {
                        taken = atomicAdd(bucket.counter, 1);
                    }
                    next = nth(WAVES + __builtin_amdgcn_readfirstlane(taken));
                } else {
                    // (a group of three tiles is the last one)
                    const int32_t first = alone(unit) ? p.column_tiles - 3 : unit.tile - wave % unit.step;
                    if (alone(unit) && unit.tile < first + 2) {
                        next.tile++;
                    } else {
                        next.node += WAVES / unit.step;
                        next.tile = alone(unit) ? first : unit.tile;
                        if (next.node >= (unit.step == 3 && wave < 3 ? last_quarter : node1)) {
                            next = begin_tiles(first + unit.step);
                        }
                    }
                }
                const int32_t after = exists(next) ? begin_of(next.node) : 0;
                tile = unit.tile;
                columns_of.set_tile(tile);
                clear();
                do {
                    n = min(WAVE, begin_of(unit.node + 1) - at);
                    add_up(here, at, n, n == WAVE ? at + n : after);
                    at += n;
                } while (n == WAVE);
                finish(unit.node);
                unit = next;
                at = after;
            }
        } else {
            int32_t at = LISTS == ORDERED ? begin_of(node0) : lower_bound(p.sorted, p.n_edges, node0, lane), n;
            Positions here = positions(at);
            for (int32_t node = node0; node < node1; node++) {
                clear();
                do {
                    if constexpr (LISTS == SEGMENTS) {
                        const unsigned long long others = __ballot(!here.inside || here.name != node);
                        n = others == 0 ? WAVE : __ffsll(others) - 1;
                    } else {
                        n = min(WAVE, begin_of(node + 1) - at);
                    }
                    add_up(here, at, n, at + n);
                    at += n;
                } while (n == WAVE);
                finish(node);
            }
        }
    }
}

template <typename T, int N, int COLUMNS, Lists LISTS, bool SHARED>
__global__ __launch_bounds__(THREADS)
__attribute__((amdgpu_waves_per_eu(contract_waves<T, N, COLUMNS>()))) void contract_kernel(const ContractArgs<T> args) {
    extern __shared__ __align__(16) char lds[];
    int32_t block = blockIdx.x;
    if constexpr (LISTS == BUCKETS) {
        const int32_t blocks = args.walk.ranges * (SHARED ? args.walk.column_tiles : 1);
        block = swizzled(block, blocks);
        if (block >= blocks) {
            return;
        }
    }
    contract<T, N, COLUMNS, LISTS, SHARED>(args, lds, block);
}

// ---------------------------------------------------------------- gradients --
template <typename T> struct EdgeArgs {
    Walk<T> walk;
    const T* grad_output; // [n_nodes][n_out][L]
    T* grad_A;            // [n_edges][nA], may be null
    T* grad_B;            // [n_edges][L], may be null
    int32_t shares;       // wavefronts per node, each with a share of its edges (0: a share of all edges)
    int32_t late, less;   // the first `late` shares of all edges have `less` edges less than the others
};

/// How a wavefront shares out its lanes: several edges side by side where G fits the registers of a lane.
template <int N, int COLUMNS> using EdgeSums = Sums<N, COLUMNS, N == 16 ? 1 : WAVE / COLUMNS>;
/// Wavefronts per SIMD.
template <typename T, int N, int COLUMNS> constexpr int edge_waves() {
    constexpr int REGISTERS = (N * EdgeSums<N, COLUMNS>::M2 + N + 44) * static_cast<int>(sizeof(T)) / 4;
    return REGISTERS <= 100 ? 4 : REGISTERS <= 140 ? 3 : 2;
}
template <typename T, int N, int COLUMNS> constexpr size_t edge_lds() {
    using S = EdgeSums<N, COLUMNS>;
    return table_slots<S, true>() * sizeof(T) +
           std::max(table_slots<S, true>() * sizeof(int32_t), WAVES * S::TILES * 16 * pitch<COLUMNS>() * sizeof(T));
}

template <typename T, int N, int COLUMNS>
__device__ __forceinline__ void edge_gradients(const EdgeArgs<T>& args, char* lds, const int32_t block) {
    using M = Mfma<T>;
    using S = EdgeSums<N, COLUMNS>;
    constexpr int EDGES = S::EDGES, M2 = S::M2, PITCH = pitch<COLUMNS>(), STAGE = S::TILES * 16 * PITCH;
    const Walk<T>& p = args.walk;
    T* table = reinterpret_cast<T*>(lds);
    T* stages = table + table_slots<S, true>();
    int32_t* owner = reinterpret_cast<int32_t*>(stages); // (while the table is built)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE); // (uniform, and known to be)
    T* stage = stages + wave * STAGE;

    Columns<T, S> columns_of(p);
    const int lane = columns_of.lane;
    build<T, S, true>(table, owner, p.C, p.table, [] {});

    const int32_t range = block * WAVES + wave;
    if (range >= p.ranges) {
        return;
    }
    int32_t first = 0, n_all = p.n_edges, share = range, shares = p.ranges;
    if (args.shares > 0) {
        share = range % args.shares;
        shares = args.shares;
        int32_t last;
        bounds_of(p.sorted, p.n_edges, range / args.shares, lane, first, last);
        n_all = last - first;
    }
    auto begin_of = [&](int32_t which) {
        const int32_t less = args.less * min(which, args.late);
        return first + static_cast<int32_t>((static_cast<int64_t>(n_all) + args.less * args.late) * which / shares) - less;
    };
    const int32_t begin = begin_of(share), end = begin_of(share + 1);
    BufferOf<T> G;
    const uint32_t g_block_bytes = static_cast<uint32_t>(p.table.n_out) * columns_of.row_bytes;
    G.set(args.grad_output, static_cast<uint32_t>(p.n_blocks) * g_block_bytes);
    const int row16 = lane >> 4, sub = lane & 15;
    constexpr int FOLDED = (N + 3) / 4;
    // (with registers to spare for grad_output and the operands at once)
    constexpr bool MEANWHILE = N * M2 * sizeof(T) <= 400;
    constexpr uint32_t A_ROW_BYTES = N * sizeof(T);
    // the component of A whose gradient ends up in this lane, and where in an edge's (or EDGES edges') rows it goes
    const bool bit[4] = {(lane & 8) != 0, (lane & 4) != 0, (lane & 2) != 0, (lane & 1) != 0};
    const int32_t of_row = bit[0] + 2 * bit[1] + 4 * bit[2];
    const int32_t component = EDGES == 1      ? 4 * sub + ((row16 & 1) << 1 | row16 >> 1)
                              : COLUMNS == 32 ? 2 * of_row + (row16 & 1)
                                              : of_row + 8 * bit[3];
    const bool holds = component < N && (EDGES == 1 ? sub < FOLDED : COLUMNS == 16 || !bit[3]);
    const uint32_t a_at =
        static_cast<uint32_t>(columns_of.slot * N + component) * static_cast<uint32_t>(sizeof(T)) | unless(holds);
    // (a gradient that is not wanted: a tensor of no bytes, which stores do not reach)
    BufferOf<T> to_A, to_B;
    to_A.set(args.grad_A, args.grad_A != nullptr ? static_cast<uint32_t>(p.n_edges) * A_ROW_BYTES : 0);
    to_B.set(args.grad_B, args.grad_B != nullptr ? static_cast<uint32_t>(p.n_edges) * columns_of.row_bytes : 0);
    BufferOf<T> A, rows; // (EDGES > 1)
    A.set(p.A, static_cast<uint32_t>(p.n_edges) * A_ROW_BYTES);
    rows.set(p.rows, static_cast<uint32_t>(p.n_blocks) * columns_of.block_bytes);
    const T* spread_from = stage + columns_of.part * S::VALUES * PITCH + columns_of.c;

    for (int32_t tile = 0; tile < p.column_tiles; tile++) {
        columns_of.set_tile(tile);
        // what this lane stores of an edge's gradients, if anything: an element of grad_B, and a
        // component of grad_A, to which the columns of the tiles before are added
        const uint32_t b_at = (static_cast<uint32_t>(columns_of.slot) * columns_of.row_bytes + columns_of.column_bytes) |
                              unless(columns_of.part == 0 && columns_of.column_inside);
        BufferOf<T> from_A;
        from_A.set(args.grad_A, tile == 0 || args.grad_A == nullptr ? 0 : static_cast<uint32_t>(p.n_edges) * A_ROW_BYTES);
        int32_t at = begin;
        Window<T> window(p, at, lane);
        while (at < end) {
            const int32_t node = __builtin_amdgcn_readfirstlane(window.receiver);
            T g[N * M2];
            // G = D^T grad_output of the node, MC components of A at a time through LDS; grad_output is asked
            // for before, and G made while, the operands of the first edges are on their way
            const bool exists = in_bounds(node, p.n_blocks);
            T upstream[COLUMNS / 16][4];
#pragma unroll
            for (int t = 0; t < COLUMNS / 16; t++) {
#pragma unroll
                for (int s3 = 0; s3 < 4; s3++) {
                    const int32_t o = 4 * s3 + row16, column = tile * COLUMNS + 16 * t + sub;
                    upstream[t][s3] = G.load(
                        (static_cast<uint32_t>(node) * g_block_bytes + static_cast<uint32_t>(o) * columns_of.row_bytes +
                         static_cast<uint32_t>(column) * static_cast<uint32_t>(sizeof(T))) |
                            unless(exists && o < p.table.n_out && column < p.L),
                        0
                    );
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            auto spread = [&] {
#pragma unroll
                for (int chunk = 0; chunk < S::CHUNKS; chunk++) {
#pragma unroll
                    for (int zt = 0; zt < S::TILES; zt++) {
                        typename M::Acc acc[COLUMNS / 16];
#pragma unroll
                        for (int t = 0; t < COLUMNS / 16; t++) {
                            acc[t] = M::zero();
                        }
#pragma unroll
                        for (int s3 = 0; s3 < 4; s3++) {
                            if (4 * s3 < p.table.n_out) { // (uniform)
                                const T left = table[((chunk * S::TILES + zt) * 4 + s3) * WAVE + lane];
#pragma unroll
                                for (int t = 0; t < COLUMNS / 16; t++) {
                                    acc[t] = M::mma(left, upstream[t][s3], acc[t]);
                                }
                            }
                        }
#pragma unroll
                        for (int t = 0; t < COLUMNS / 16; t++) {
#pragma unroll
                            for (int r = 0; r < 4; r++) {
                                stage[(zt * 16 + M::row(lane, r)) * PITCH + 16 * t + sub] = acc[t][r];
                            }
                        }
                    }
                    wave_sync();
#pragma unroll
                    for (int k = 0; k < S::VALUES; k++) {
                        if (chunk * S::VALUES + k < N * M2) {
                            g[chunk * S::VALUES + k] = spread_from[k * PITCH];
                        }
                    }
                    wave_sync();
                }
                if constexpr (!S::EXACT) { // (what the last part has no row for)
#pragma unroll
                    for (int i = 0; i < N; i++) {
                        g[i * M2 + M2 - 1] = columns_of.has_row(M2 - 1) ? g[i * M2 + M2 - 1] : T(0);
                    }
                }
            };
            auto gradients = [&](int32_t first) {
                return [&, first](const T (&a)[N], const auto& operands, int32_t k) {
                    T u[N];
#pragma unroll
                    for (int i = 0; i < N; i++) {
                        u[i] = g[i * M2] * operands.w[0];
#pragma unroll
                        for (int m = 1; m < M2; m++) {
                            u[i] += g[i * M2 + m] * operands.w[m];
                        }
                    }
                    const uint32_t edge = static_cast<uint32_t>(first + k);
                    T sum = a[0] * u[0];
#pragma unroll
                    for (int i = 1; i < N; i++) {
                        sum += a[i] * u[i];
                    }
                    // over the parts: rows of 16 lanes, or halves
                    if constexpr (S::PARTS == 4) {
                        sum = sum_rows(sum, sum);
                    }
                    if constexpr (S::PARTS > 1) {
                        sum = sum_halves(sum, sum);
                    }
                    to_B.store(sum, b_at, edge * columns_of.row_bytes);
                    const T b = columns_of.column_inside ? operands.b : T(0);
                    auto term = [&](int i) { return i < N ? u[i < N ? i : 0] * b : T(0); };
                    // the sum over columns and parts: four values folded together across the halves
                    // and the rows of the wavefront, so that a row of 16 lanes sums one
                    T mine = T(0);
#pragma unroll
                    for (int i = 0; i < FOLDED; i++) {
                        const T low = sum_halves(term(4 * i), term(4 * i + 1));
                        const T folded =
                            sum_of_row(sum_rows(low, 4 * i + 2 < N ? sum_halves(term(4 * i + 2), term(4 * i + 3)) : T(0)));
                        mine = sub == i ? folded : mine;
                    }
                    to_A.store(mine + operands.more, a_at, edge * A_ROW_BYTES);
                };
            };
            // (EDGES > 1: of the lane's edge)
            auto gradients_of_its_own = [&](const auto& operands, uint32_t edge, bool valid) {
                const T b = columns_of.column_inside ? operands.b : T(0);
                T sum = T(0), term[N];
                unrolled(std::make_integer_sequence<int, N>{}, [&](auto i) {
                    T u = g[i * M2] * operands.w[0];
#pragma unroll
                    for (int m = 1; m < M2; m++) {
                        u += g[i * M2 + m] * operands.w[m];
                    }
                    term[i] = u * b;
                    sum += rotated<0x150 + i>(operands.a) * u; // (row_newbcast: element i of the row of A)
                });
                const uint32_t lost = unless(valid);
                to_B.store(sum, b_at | lost, edge * columns_of.row_bytes);
                to_A.store(folded<COLUMNS, N>(term, bit) + operands.more, a_at | lost, edge * A_ROW_BYTES);
            };
            bool spread_out = false;
            if constexpr (!MEANWHILE) {
                if (exists) {
                    spread();
                    spread_out = true;
                }
            }
            auto spread_once = [&] {
                if (MEANWHILE && !spread_out) { // (uniform)
                    spread();
                    spread_out = true;
                }
            };
            int32_t n;
            do {
                n = min(window.edges_of(node), end - at);
                const Window<T> next(p, at + n, lane);
                if constexpr (EDGES > 1) {
                    if (exists && n > 0) {
                        columns_of.side_by_side(
                            A, rows, window.source, at, n,
                            [&](auto& operands, uint32_t edge) { operands.more = from_A.load(a_at, edge * A_ROW_BYTES); },
                            spread_once, gradients_of_its_own
                        );
                    }
                } else if (exists && n > 0) {
                    const int32_t first = at;
                    columns_of.template over<1>(
                        window.source, n, [&](int32_t k) { return first + k; },
                        [&](auto& operands, int32_t k) {
                            operands.more = from_A.load(a_at, static_cast<uint32_t>(first + k) * A_ROW_BYTES);
                        },
                        spread_once, gradients(first)
                    );
                }
                at += n;
                window = next;
            } while (n == WAVE);
        }
    }
}

/// The first plan.shares workgroups split `senders` before their part of the edges, which is the smaller for it.
template <typename T, int N, int COLUMNS>
__global__ __launch_bounds__(THREADS)
__attribute__((amdgpu_waves_per_eu(edge_waves<T, N, COLUMNS>()))) void
edge_kernel(const EdgeArgs<T> args, const Shares shares, const SharePlan plan, const int32_t* __restrict__ senders) {
    extern __shared__ __align__(16) char lds[];
    if (static_cast<int32_t>(blockIdx.x) < plan.shares) { // (uniform)
        split_share<THREADS>(reinterpret_cast<int32_t*>(lds), shares, plan, senders, blockIdx.x);
        __syncthreads();
    }
    edge_gradients<T, N, COLUMNS>(args, lds, blockIdx.x);
}

template <typename T, int N, int COLUMNS> constexpr int small_waves() {
    return std::min(contract_waves<T, N, COLUMNS>(), edge_waves<T, N, COLUMNS>());
}

/// All gradients of a small graph in one launch: the first `nodes` workgroups have a node and a tile of
/// columns of grad_W each, and look through the index for its edges themselves; the others grad_A and grad_B.
/// Bound by the launch and one chain of loads. Against the listing of the edges, grad_A and grad_B, and grad_W
/// one after the other, 9 components, 32 columns, f32 / f64: 600 edges 24.0 -> 11.8 / 26.6 -> 12.8 us, 5000 edges
/// of 200 nodes 27.0 -> 14.9 / 31.3 -> 17.0.
template <typename T, int N, int COLUMNS>
__global__ __launch_bounds__(THREADS)
__attribute__((amdgpu_waves_per_eu(small_waves<T, N, COLUMNS>()))) void
small_kernel(const ContractArgs<T> of_nodes, const EdgeArgs<T> of_edges, int32_t nodes) {
    extern __shared__ __align__(16) char lds[];
    if (static_cast<int32_t>(blockIdx.x) < nodes) { // (uniform)
        contract<T, N, COLUMNS, LOOKED_FOR, true>(of_nodes, lds, blockIdx.x);
    } else {
        edge_gradients<T, N, COLUMNS>(of_edges, lds, blockIdx.x - nodes);
    }
}

// --------------------------------------------------------------------- host --
/// What a tile of columns costs: the multiply-adds of a lane, and some eight
/// instructions' worth of everything else.
template <int N, int COLUMNS> constexpr int cost() { return (N + 1) * Sums<N, COLUMNS>::M2 + 8; }

/// Workgroups of a sum on the device at a time.
template <typename T, int N, int COLUMNS> int64_t resident_sums() {
    return static_cast<int64_t>(compute_units()) * contract_waves<T, N, COLUMNS>();
}

/// body(N, COLUMNS): the cheapest tiles. EDGES: for the gradients by edge, in double of 32 columns at most for 9
/// components (60 000 edges, 64 columns, grad_A and grad_B with 64 / 32 at a time 66 / 56 us, 300 000 259 / 248; in float
/// 31 / 37 and 128 / 132). `more`: what a tile costs beside that.
enum Of { EDGES, SUMS, BUCKETED };
template <typename T, Of OF, typename Body> void with_layout(const Shape& s, Body&& body, int more = 0) {
    auto with_columns = [&](auto n) {
        constexpr int N = decltype(n)::value;
        // (sums that fit the registers of a lane)
        constexpr int MOST = N == 16                            ? (sizeof(T) == 4 ? 32 : 16)
                             : OF == EDGES && N == 9 && sizeof(T) == 8 ? 32
                                                                 : 64;
        int best = 16, least = (s.L + 15) / 16 * (cost<N, 16>() + more);
        if (const int c = (s.L + 31) / 32 * (cost<N, 32>() + more); MOST >= 32 && c <= least) {
            best = 32;
            least = c;
        }
        if (const int c = (s.L + 63) / 64 * (cost<N, 64>() + more); MOST >= 64 && c <= least) {
            best = 64;
        }
        // The sums of few nodes take more, narrower tiles, which are wavefronts of their own. Where a workgroup gathers a
        // bucket first, it is better used for a node and all of the columns that fit its registers, if no more nodes
        // than run at a time leave it a node to itself (grad_W with grad_A and grad_B, 9 components, f32: 30 000 edges of
        // 1000 nodes, 32 columns, 16 / 32 at a time 40.3 / 35.3 us; of 600, 64 columns, 50.9 / 44.6; but 9000 of 300 in
        // double 46.8 / 51.7).
        const int64_t nodes = s.n_nodes;
        const bool wide = OF == BUCKETED && best > 16 && nodes * ((s.L + 15) / 16) > resident_sums<T, N, 16>() &&
                          (best == 32   ? nodes * ((s.L + 31) / 32) <= resident_sums<T, N, MOST >= 32 ? 32 : 16>()
                           : sizeof(T) == 4 ? nodes * ((s.L + 63) / 64) <= resident_sums<T, N, MOST >= 64 ? 64 : 16>()
                                            : false);
        if (OF != EDGES && !wide && nodes * ((s.L + best - 1) / best) < 4 * compute_units()) {
            best = 16;
        }
        if (best == 16) {
            body(n, std::integral_constant<int, 16>{});
        }
        if constexpr (MOST >= 32) {
            if (best == 32) {
                body(n, std::integral_constant<int, 32>{});
            }
        }
        if constexpr (MOST >= 64) {
            if (best == 64) {
                body(n, std::integral_constant<int, 64>{});
            }
        }
    };
    if (s.nA == 4) {
        with_columns(std::integral_constant<int, 4>{});
    } else if (s.nA == 9) {
        with_columns(std::integral_constant<int, 9>{});
    } else {
        with_columns(std::integral_constant<int, 16>{});
    }
}

template <typename Kernel> void allow_lds(Kernel kernel, size_t lds) {
    if (lds > 64 * 1024) {
        MOPS_HIP_CHECK(hipFuncSetAttribute(
            reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)
        ));
    }
}

template <typename T>
Walk<T> walk_of(
    const Shape& s, const T* A, const T* B, const T* rows, const T* C, const int32_t* sorted, const int32_t* gather,
    const Dense& table
) {
    Walk<T> w{};
    w.A = A;
    w.B = B;
    w.rows = rows;
    w.C = C;
    w.n_edges = s.n_edges;
    w.n_blocks = s.n_nodes;
    w.L = s.L;
    w.sorted = sorted;
    w.gather = gather;
    w.table = table;
    return w;
}

template <typename T, Lists LISTS> void contract(ContractArgs<T> args, const Shape& s, hipStream_t stream) {
    with_layout<T, LISTS == BUCKETS ? BUCKETED : SUMS>(s, [&](auto n, auto columns) {
        constexpr int N = decltype(n)::value, COLUMNS = decltype(columns)::value;
        Walk<T>& w = args.walk;
        const size_t lds = LISTS == BUCKETS ? contract_lds<T, N, COLUMNS>(args.plan.per_bucket) : contract_lds<T, N, COLUMNS>();
        w.column_tiles = (s.L + COLUMNS - 1) / COLUMNS;
        auto launch = [&](auto kernel, int64_t ranges, int waves_per_range) {
            w.ranges = static_cast<int32_t>(std::min<int64_t>(s.n_nodes, std::max<int64_t>(1, ranges)));
            const int32_t blocks = static_cast<int32_t>(ceil_div(static_cast<size_t>(w.ranges) * waves_per_range, WAVES));
            allow_lds(kernel, lds);
            kernel<<<LISTS == BUCKETS ? swizzled_blocks(blocks) : blocks, THREADS, lds, stream>>>(args);
        };
        const int64_t resident = resident_sums<T, N, COLUMNS>();
        const bool shared = static_cast<int64_t>(s.n_nodes) * w.column_tiles <= resident;
        if (shared) {
            launch(contract_kernel<T, N, COLUMNS, LISTS, true>, s.n_nodes, WAVES * w.column_tiles);
        } else if (LISTS == BUCKETS) {
            launch(contract_kernel<T, N, COLUMNS, LISTS, false>, args.plan.buckets, WAVES);
        } else {
            launch(contract_kernel<T, N, COLUMNS, LISTS, false>, resident * WAVES / w.column_tiles, w.column_tiles);
        }
    });
    MOPS_HIP_CHECK(hipGetLastError());
}

} // namespace

bool covers(int32_t nA, int32_t block_rows, int32_t result_rows) {
    return (nA == 4 || nA == 9 || nA == 16) && block_rows == nA && result_rows <= MAX_INDEX;
}

template <typename T>
void forward(
    T* output, const T* A, const T* B, const T* C, const T* W, const Indices& indices, const Shape& s, hipStream_t stream
) {
    ContractArgs<T> args{};
    args.walk = walk_of(
        s, A, B, W, C, indices.output_1, indices.W_1, Dense{indices.A, indices.W_2, indices.output_2, s.N, s.n3}
    );
    args.result = output;
    MainKernelTimer timer(stream);
    contract<T, SEGMENTS>(args, s, stream);
}

namespace {

template <typename T>
ContractArgs<T> of_senders(
    T* grad_W, const T* grad_output, const T* A, const T* B, const T* C, const Indices& indices, const Shape& s
) {
    ContractArgs<T> args{};
    args.walk = walk_of<T>(
        s, A, B, grad_output, C, nullptr, indices.output_1, Dense{indices.A, indices.output_2, indices.W_2, s.N, s.n2}
    );
    args.result = grad_W;
    args.senders = indices.W_1;
    return args;
}

template <typename T>
EdgeArgs<T> of_edges(
    T* grad_A, T* grad_B, const T* grad_output, const T* A, const T* B, const T* C, const T* W, const Indices& indices,
    const Shape& s
) {
    EdgeArgs<T> args{};
    args.walk = walk_of(
        s, A, B, W, C, indices.output_1, indices.W_1, Dense{indices.A, indices.W_2, indices.output_2, s.N, s.n3}
    );
    args.grad_output = grad_output;
    args.grad_A = grad_A;
    args.grad_B = grad_B;
    return args;
}

/// The wavefronts' shares of the edges; returns the workgroups that takes.
template <typename T, int N, int COLUMNS> size_t share_out(EdgeArgs<T>& args, const Shape& s) {
    Walk<T>& w = args.walk;
    w.column_tiles = (s.L + COLUMNS - 1) / COLUMNS;
    const int64_t resident = static_cast<int64_t>(compute_units()) * 4 * edge_waves<T, N, COLUMNS>();
    // Every wavefront has as many edges as the next, whatever nodes they are of, and makes G of each
    // (against a range of nodes each, 9 components, 32 columns, f32 / f64, whole vjp: 60 000 edges of 2000
    // nodes 74 -> 69 us in double, 200 000 of 6600 134 -> 125 / 212 -> 195; 91 000 of 3000, 16 components,
    // 64 columns, 239 -> 219 / 464 -> 398). Where two wavefronts or more share a node, with four edges each
    // at least, that is only more of G (600 edges of 20 nodes, listing and grad_W with it, 24.0 -> 24.8; for 16 components in float, of
    // which G is the most work, also with one: 50 000 of 2000 85.2 -> 87.1).
    const int64_t shares = std::min<int64_t>(s.n_edges / (4 * static_cast<int64_t>(s.n_nodes)), resident / s.n_nodes);
    // Shares of four edges or more, but of two where nodes have fewer than four each (a G for every one of
    // them, one after the other: 400 edges of 300 nodes, whole vjp, f32 / f64 16.8 -> 11.7 / 20.4 -> 14.6 us, 2000 of 1500
    // 36.3 -> 30.1 in double, 3000 of 1000, 16 components, 45.1 -> 40.3 in float).
    const int64_t least = N == 16 && sizeof(T) == 4 ? 1 : 2;
    const int64_t of_all = std::max<int64_t>(s.n_edges / 4, std::min(s.n_edges / 2, s.n_nodes));
    args.shares = shares >= least ? static_cast<int32_t>(shares) : 0;
    w.ranges = static_cast<int32_t>(shares >= least ? s.n_nodes * shares : std::max<int64_t>(1, std::min(of_all, resident)));
    return ceil_div(static_cast<size_t>(w.ranges), WAVES);
}

} // namespace

template <typename T> SenderLists plan_lists(const Shape& s) {
    SenderLists lists{};
    with_layout<T, BUCKETED>(s, [&](auto n, auto columns) {
        constexpr int N = decltype(n)::value, COLUMNS = decltype(columns)::value;
        const int32_t tiles = (s.L + COLUMNS - 1) / COLUMNS;
        const int64_t resident = resident_sums<T, N, COLUMNS>();
        // A node by a workgroup for each of its tiles if there are no more of them than run at a time; else as many
        // buckets as workgroups run at a time (fewer would leave some idle), or twice or four times as many.
        const bool shared = static_cast<int64_t>(s.n_nodes) * tiles <= resident;
        // (of few nodes no more buckets than leave each wavefront a node and tile: grad_W alone, 10 000 edges of 1000 nodes,
        // 16 components, f32, with a bucket per two nodes / per four 25.6 / 21.9 us, 9 in double 22.5 / 20.1)
        const int64_t units = static_cast<int64_t>(s.n_nodes) * std::min(tiles, WAVES);
        for (int64_t buckets = shared ? s.n_nodes : std::min<int64_t>(resident, (units + WAVES - 1) / WAVES);
             buckets <= MOST_SHARE_BUCKETS && !lists.in_shares; buckets *= 2) {
            lists.in_shares = plan_shares(lists.plan, s.n_nodes, s.n_edges, static_cast<int32_t>(buckets));
        }
        lists.copies = shared ? tiles : 1;
    });
    return lists;
}

template <typename T>
void weight_gradient(
    T* grad_W, const T* grad_output, const T* A, const T* B, const T* C, const Indices& indices, const Shape& s,
    const SenderLists* lists, void* workspace, const EdgesBySender* ordered, hipStream_t stream
) {
    ContractArgs<T> args = of_senders(grad_W, grad_output, A, B, C, indices, s);
    if (lists != nullptr) {
        args.plan = lists->plan;
        args.shares = shares_in(workspace, lists->plan);
        contract<T, BUCKETS>(args, s, stream);
    } else {
        args.ordered = *ordered;
        contract<T, ORDERED>(args, s, stream);
    }
}

template <typename T>
void edge_gradients(
    T* grad_A, T* grad_B, const T* grad_output, const T* A, const T* B, const T* C, const T* W, const Indices& indices,
    const Shape& s, const SenderLists* lists, void* workspace, hipStream_t stream
) {
    EdgeArgs<T> args = of_edges(grad_A, grad_B, grad_output, A, B, C, W, indices, s);
    SharePlan plan{};
    Shares shares{};
    if (lists != nullptr) {
        plan = lists->plan;
        shares = shares_in(workspace, plan);
    }
    MainKernelTimer timer(stream);
    with_layout<T, EDGES>(s, [&](auto components, auto columns) {
        constexpr int N = decltype(components)::value, COLUMNS = decltype(columns)::value;
        const size_t lds =
            std::max(edge_lds<T, N, COLUMNS>(), split_lds<THREADS>(plan.buckets) * sizeof(int32_t));
        const size_t blocks = std::max(share_out<T, N, COLUMNS>(args, s), static_cast<size_t>(plan.shares));
        if (args.shares == 0) {
            // (splitting 1024 edges takes as long as some six edges of a wavefront's part, 4096 as 18)
            args.late = std::min(plan.shares * WAVES, args.walk.ranges);
            args.less = std::min(2 + plan.share / 256, s.n_edges / args.walk.ranges / 2);
        }
        auto kernel = edge_kernel<T, N, COLUMNS>;
        allow_lds(kernel, lds);
        kernel<<<static_cast<unsigned>(blocks), THREADS, lds, stream>>>(args, shares, plan, indices.W_1);
    });
    MOPS_HIP_CHECK(hipGetLastError());
}

namespace {

/// What a tile costs a small graph beside its columns: tiles are one after the other for the edges' wavefronts,
/// and little else bounds it (2000 edges of 60 nodes, 40 columns, f64, with 16 / 32 at a time 18.7 / 15.5 us).
constexpr int SMALL_TILE_COST = 4;

template <typename T> bool is_small(const Shape& s) {
    bool result = false;
    with_layout<T, EDGES>(s, [&](auto n, auto columns) {
        constexpr int WAVES_PER_SIMD = small_waves<T, decltype(n)::value, decltype(columns)::value>();
        const int32_t tiles = (s.L + decltype(columns)::value - 1) / decltype(columns)::value;
        const int64_t resident = static_cast<int64_t>(compute_units()) * WAVES_PER_SIMD; // workgroups
        const int32_t edges = thresholds::COLUMNS_EDGES_AS_THEY_ARE;
        result = s.n_edges <= (s.nA < 16 ? edges : sizeof(T) == 4 ? edges / 4 * 3 : edges / 2) &&
                 static_cast<int64_t>(s.n_nodes) * tiles <= resident;
    }, SMALL_TILE_COST);
    return result;
}

} // namespace

bool small(const Shape& s, size_t element_size) { return element_size == 4 ? is_small<float>(s) : is_small<double>(s); }

template <typename T>
void small_vjp(
    T* grad_A, T* grad_B, T* grad_W, const T* grad_output, const T* A, const T* B, const T* C, const T* W,
    const Indices& indices, const Shape& s, hipStream_t stream
) {
    ContractArgs<T> nodes = of_senders(grad_W, grad_output, A, B, C, indices, s);
    EdgeArgs<T> edges = of_edges(grad_A, grad_B, grad_output, A, B, C, W, indices, s);
    MainKernelTimer timer(stream);
    with_layout<T, EDGES>(s, [&](auto components, auto columns) {
        constexpr int N = decltype(components)::value, COLUMNS = decltype(columns)::value;
        constexpr size_t lds = std::max(edge_lds<T, N, COLUMNS>(), contract_lds<T, N, COLUMNS>());
        nodes.walk.column_tiles = (s.L + COLUMNS - 1) / COLUMNS;
        nodes.walk.ranges = s.n_nodes;
        const size_t of_nodes = grad_W != nullptr ? static_cast<size_t>(s.n_nodes) * nodes.walk.column_tiles : 0;
        const size_t of_edges = grad_A != nullptr || grad_B != nullptr ? share_out<T, N, COLUMNS>(edges, s) : 0;
        auto kernel = small_kernel<T, N, COLUMNS>;
        allow_lds(kernel, lds);
        kernel<<<static_cast<unsigned>(of_nodes + of_edges), THREADS, lds, stream>>>(nodes, edges, static_cast<int32_t>(of_nodes));
    }, SMALL_TILE_COST);
    MOPS_HIP_CHECK(hipGetLastError());
}

#define MOPS_INSTANTIATE(T)                                                                         \
    template void forward<T>(                                                                      \
        T*, const T*, const T*, const T*, const T*, const Indices&, const Shape&, hipStream_t      \
    );                                                                                             \
    template void edge_gradients<T>(                                                               \
        T*, T*, const T*, const T*, const T*, const T*, const T*, const Indices&, const Shape&, const SenderLists*, void*, hipStream_t \
    );                                                                                             \
    template SenderLists plan_lists<T>(const Shape&);                                              \
    template void weight_gradient<T>(                                                              \
        T*, const T*, const T*, const T*, const T*, const Indices&, const Shape&, const SenderLists*, void*, const EdgesBySender*, hipStream_t \
    );                                                                                             \
    template void small_vjp<T>(                                                                    \
        T*, T*, T*, const T*, const T*, const T*, const T*, const T*, const Indices&, const Shape&, hipStream_t \
    );
MOPS_INSTANTIATE(float)
MOPS_INSTANTIATE(double)
#undef MOPS_INSTANTIATE

} // namespace mops::amd::sasaw_columns
