// Homogeneous polynomial evaluation with many monomials or many features, for
// gfx950 (semantics: hpe.hip).
//
// A workgroup keeps the values of R = 4 V rows in LDS, feature by feature, the
// R values of a feature side by side (and one feature more, all zero, that
// stands for an index outside the tensor). Its 1024 threads are 256 teams of
// four lanes; a team works on one monomial at a time for all R rows, a lane
// holding V of them: a factor is then 16 V sizeof(T) / 4 consecutive bytes of
// LDS, read by 16-byte loads. Four monomials are loaded at a time, one by each
// lane of the team, and handed round by DPP (the add that makes the LDS
// address takes the offset of the team's other lane as its operand), so the
// table costs an instruction per factor and no scalar loads.
//
// What bounds these kernels is LDS: order (forward) or order * (order - 1)
// (gradients) values per row and monomial, and that the features which a pass of 16-byte
// reads brings for four teams are as often as not on the same quarter of the banks (of
// 1000 rows, 2000 features, 100 000 monomials of order 4, float, 0.48 of the gradients' 71 us
// of LDS are such conflicts; the best order of a record's factors would leave nine tenths
// of that time, the best places of four records as well four fifths). A term of a gradient reads the
// order - 1 OTHER factors and adds up in registers; nothing is added in LDS.
// For that the table is first turned round (feature -> the terms it is a
// factor of, `records_kernel`), deterministically and without atomics on
// shared counters: a stable counting sort (5 us for the counts and 24 for
// the records of 400 000 factors).
//
// 1000 rows, 2000 features, 100 000 monomials of order 4, whole calls: forward
// 91 -> 37 us (float), 98 -> 61 (double), of which LDS at 128 bytes per clock
// and compute unit needs 20 and 41; vjp 8050 -> 118 and 18 560 -> 207 (61 and
// 122); second order 1.46 s -> 414 us and 1.54 s -> 816 us, against the kernels
// that keep the accumulators of a few features, or nothing, in LDS.
#include <algorithm>
#include <type_traits>

#include "hpe_tiles.hpp"

#include "device_common.hpp"
#include "runtime.hpp"

namespace mops::amd {
namespace hpe_tiles {
namespace {

constexpr int THREADS = 1024;
constexpr int WAVES = THREADS / WAVE;
constexpr int TEAM = 4;
constexpr int TEAMS = THREADS / TEAM;
constexpr size_t LDS_LIMIT = 156 * 1024; // of the 160 KB of a compute unit
constexpr int MOST_VALUES = 4;           // per lane: one 16-byte load of floats, two of doubles

/// Values of T that one LDS load of a lane brings: V of them, 16 bytes at most.
template <typename T, int V> constexpr int chunk_values() { return V * sizeof(T) < 16 ? V : 16 / sizeof(T); }

/// Row (of the tile) that value v of lane `q` of a team stands for. `swap`
/// exchanges the two halves of a lane's values, see Tile.
template <typename T, int V> __device__ __forceinline__ int row_of(int q, int v, bool swap) {
    constexpr int E = chunk_values<T, V>();
    const int chunk = (v / E) ^ (V / E == 2 && swap ? 1 : 0);
    return chunk * (TEAM * E) + q * E + v % E;
}

/// Four-lane broadcast of lane `FROM` of every team.
template <int FROM> __device__ __forceinline__ uint32_t from_lane(uint32_t value) {
    constexpr int control = FROM | FROM << 2 | FROM << 4 | FROM << 6;
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(value), control, 0xf, 0xf, true));
}
template <int FROM> __device__ __forceinline__ float from_lane(float value) {
    return __uint_as_float(from_lane<FROM>(__float_as_uint(value)));
}
template <int FROM> __device__ __forceinline__ double from_lane(double value) {
    const uint64_t bits = static_cast<uint64_t>(__double_as_longlong(value));
    const uint64_t low = from_lane<FROM>(static_cast<uint32_t>(bits));
    const uint64_t high = from_lane<FROM>(static_cast<uint32_t>(bits >> 32));
    return __longlong_as_double(static_cast<long long>(high << 32 | low));
}

/// A monomial (forward: all its factors; gradients: the factors other than the
/// one of the list) as it lies in a lane: byte offsets of its factors in the
/// tile, and its coefficient.
template <typename T, int FACTORS> struct Term {
    uint32_t offset[FACTORS > 0 ? FACTORS : 1];
    T coefficient;
};

/// The tile in LDS. With two loads per factor and lane (four doubles) every
/// other team reads the second half first, so that the teams that are
/// served together are never all on the same half of the banks.
template <typename T, int V, int PARTS_PER_FEATURE> struct Tile {
    static constexpr int E = chunk_values<T, V>();
    static constexpr int CHUNKS = V / E;
    static constexpr int R = TEAM * V;
    static constexpr int STRIDE = PARTS_PER_FEATURE * R * static_cast<int>(sizeof(T)); // bytes per feature
    const char* lane[CHUNKS];

    __device__ __forceinline__ Tile(const char* tile, int team, int q) {
        const bool swap = CHUNKS == 2 && (team & 1) != 0;
#pragma unroll
        for (int c = 0; c < CHUNKS; c++) {
            lane[c] = tile + ((swap ? c ^ 1 : c) * TEAM + q) * E * static_cast<int>(sizeof(T));
        }
    }

    /// The V values of a feature at byte `offset`; `part`: A, or grad_grad_A behind it.
    __device__ __forceinline__ void read(T (&value)[V], uint32_t offset, int part = 0) const {
        typedef T Chunk __attribute__((ext_vector_type(E)));
#pragma unroll
        for (int c = 0; c < CHUNKS; c++) {
            const Chunk loaded =
                *reinterpret_cast<const Chunk*>(lane[c] + offset + part * R * static_cast<int>(sizeof(T)));
#pragma unroll
            for (int e = 0; e < E; e++) {
                value[c * E + e] = loaded[e];
            }
        }
    }
};
template <typename T, int PARTS_PER_FEATURE> struct Tile<T, 1, PARTS_PER_FEATURE> {
    static constexpr int R = TEAM;
    static constexpr int STRIDE = PARTS_PER_FEATURE * R * static_cast<int>(sizeof(T));
    const char* lane;
    __device__ __forceinline__ Tile(const char* tile, int, int q) : lane(tile + q * sizeof(T)) {}
    __device__ __forceinline__ void read(T (&value)[1], uint32_t offset, int part = 0) const {
        value[0] = *reinterpret_cast<const T*>(lane + offset + part * R * static_cast<int>(sizeof(T)));
    }
};

/// The rows of `source` (n_rows x nA) from row0 on into part `part` of the
/// tile, and zeros for the feature nA. A wavefront takes 16 features at a time
/// of all rows: its loads are 16 consecutive values of a row, its stores
/// consecutive LDS addresses.
template <typename T, int V, int PARTS_PER_FEATURE>
__device__ __forceinline__ void
stage(char* tile, int part, const T* __restrict__ source, int32_t row0, int32_t n_rows, int32_t nA) {
    using Layout = Tile<T, V, PARTS_PER_FEATURE>;
    constexpr int FEATURES = WAVE / TEAM;
    constexpr int AHEAD = V == 4 ? 4 : 8; // groups of features asked for together
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const int q = lane & (TEAM - 1), sub = lane / TEAM;
    const T* rows[V];
#pragma unroll
    for (int v = 0; v < V; v++) {
        rows[v] = source + static_cast<size_t>(min(row0 + row_of<T, V>(q, v, false), n_rows - 1)) * nA;
    }
    char* to = tile + part * Layout::R * sizeof(T);
    for (int32_t f0 = wave * FEATURES; f0 < nA; f0 += AHEAD * WAVES * FEATURES) {
        T value[AHEAD][V];
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            const int32_t f = min(f0 + u * WAVES * FEATURES + sub, nA - 1);
#pragma unroll
            for (int v = 0; v < V; v++) {
                value[u][v] = rows[v][f];
            }
        }
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            const int32_t f = f0 + u * WAVES * FEATURES + sub;
            if (f < nA) {
#pragma unroll
                for (int v = 0; v < V; v++) {
                    *reinterpret_cast<T*>(to + f * Layout::STRIDE + row_of<T, V>(q, v, false) * sizeof(T)) = value[u][v];
                }
            }
        }
    }
    if (threadIdx.x < Layout::R) {
        *reinterpret_cast<T*>(to + nA * Layout::STRIDE + threadIdx.x * sizeof(T)) = T(0);
    }
}

/// Adds up the V values of every lane over the teams of a workgroup, in a
/// fixed order; the sum of row r comes back in thread r < R. `exchange`:
/// WAVES * R values of LDS that nobody else uses.
template <typename T, int V> __device__ __forceinline__ T sum_over_teams(T (&value)[V], T* exchange) {
    constexpr int R = TEAM * V;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const bool swap = ((lane / TEAM) & 1) != 0;
    // (a team that reads the halves the other way round holds them the other way round)
    if constexpr (V > 1 && V / chunk_values<T, V>() == 2) {
#pragma unroll
        for (int v = 0; v < V / 2; v++) {
            const T low = value[v], high = value[v + V / 2];
            value[v] = swap ? high : low;
            value[v + V / 2] = swap ? low : high;
        }
    }
#pragma unroll
    for (int v = 0; v < V; v++) {
#pragma unroll
        for (int step = TEAM; step < WAVE; step <<= 1) {
            value[v] += __shfl_xor(value[v], step);
        }
    }
    if (lane < TEAM) {
#pragma unroll
        for (int v = 0; v < V; v++) {
            exchange[wave * R + row_of<T, V>(lane, v, false)] = value[v];
        }
    }
    __syncthreads();
    T sum = T(0);
    if (threadIdx.x < R) {
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            sum += exchange[w * R + threadIdx.x];
        }
    }
    return sum;
}

/// result[row0 + r] = the sum over the workgroups of a tile of `mine` (given by
/// thread r < R), in the order of the workgroups: all but the last one to
/// arrive leave theirs in `partial`. Written through to memory and read from
/// there, because the workgroups of a tile need not share an L2.
template <typename T>
__device__ __forceinline__ void sum_over_groups(
    T* result, T mine, T* partial, int32_t* counter, int32_t group, int32_t groups, int R, int32_t row0, int32_t n_rows
) {
    const bool holds = static_cast<int>(threadIdx.x) < R && row0 + static_cast<int32_t>(threadIdx.x) < n_rows;
    if (groups == 1) {
        if (holds) {
            result[row0 + threadIdx.x] = mine;
        }
        return;
    }
    __shared__ int32_t arrived;
    if (static_cast<int>(threadIdx.x) < R) {
        __hip_atomic_store(partial + group * R + threadIdx.x, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        arrived = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (arrived == groups - 1) {
        if (holds) {
            T sum = T(0);
            for (int32_t g = 0; g < groups; g++) {
                sum += __hip_atomic_load(partial + g * R + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            result[row0 + threadIdx.x] = sum;
        }
        if (threadIdx.x == 0) {
            __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

/// Which tile of rows and which share of it a workgroup has: the shares of a
/// tile on one XCD (workgroups are dealt out to the eight of them in turn), so
/// that its rows come from memory once.
__device__ __forceinline__ bool my_share(int32_t tiles, int32_t groups, int32_t& tile, int32_t& group) {
    const int32_t xcd = blockIdx.x & 7, turn = blockIdx.x >> 3;
    tile = turn / groups * 8 + xcd;
    group = turn % groups;
    return tile < tiles;
}
unsigned blocks_of(const Plan& plan) { return static_cast<unsigned>((plan.tiles + 7) / 8 * 8 * plan.groups); }

// ------------------------------------------------------------------ forward --
template <typename T, int ORDER, int V>
__global__ __launch_bounds__(THREADS) void forward_kernel(
    T* output,
    T* partial,
    int32_t* counters,
    const T* __restrict__ A,
    const T* __restrict__ C,
    const int32_t* __restrict__ P,
    int32_t n_rows,
    int32_t nA,
    int32_t n_monomials,
    int32_t share, // monomials per workgroup, a multiple of TEAM
    int32_t tiles,
    int32_t groups
) {
    using Layout = Tile<T, V, 1>;
    extern __shared__ __align__(16) char lds[];
    T* exchange = reinterpret_cast<T*>(lds);
    char* tile = lds + WAVES * Layout::R * sizeof(T);
    int32_t which, group;
    if (!my_share(tiles, groups, which, group)) {
        return;
    }
    const int32_t row0 = which * Layout::R;
    const int team = threadIdx.x / TEAM, q = threadIdx.x & (TEAM - 1);
    const int32_t begin = group * share;
    const int32_t end = min(begin + share, n_monomials);

    Term<T, ORDER> next;
    auto fetch = [&](int32_t j) { // (a monomial beyond the end: zeros)
        const bool exists = j < end;
        const int32_t safe = exists ? j : n_monomials - 1;
        const int32_t* factors = P + static_cast<size_t>(safe) * ORDER;
#pragma unroll
        for (int k = 0; k < ORDER; k++) {
            next.offset[k] = static_cast<uint32_t>(exists ? factors[k] : nA);
        }
        next.coefficient = exists ? C[safe] : T(0);
    };
    int32_t j = begin + team * TEAM + q;
    fetch(j);
    stage<T, V, 1>(tile, 0, A, row0, n_rows, nA);
    __syncthreads();

    const Layout values(tile, team, q);
    T sum[V];
#pragma unroll
    for (int v = 0; v < V; v++) {
        sum[v] = T(0);
    }
    for (; j - q < end; j += TEAMS * TEAM) {
        Term<T, ORDER> now = next;
        fetch(j + TEAMS * TEAM);
#pragma unroll
        for (int k = 0; k < ORDER; k++) {
            // (as unsigned, a negative index is a large one)
            now.offset[k] = min(now.offset[k], static_cast<uint32_t>(nA)) * static_cast<uint32_t>(Layout::STRIDE);
        }
        auto one = [&](auto lane) {
            constexpr int FROM = decltype(lane)::value;
            T product[V];
            const T coefficient = from_lane<FROM>(now.coefficient);
            T factor[ORDER][V];
#pragma unroll
            for (int k = 0; k < ORDER; k++) {
                values.read(factor[k], from_lane<FROM>(now.offset[k]));
            }
#pragma unroll
            for (int v = 0; v < V; v++) {
                product[v] = coefficient;
#pragma unroll
                for (int k = 0; k < ORDER - 1; k++) {
                    product[v] *= factor[k][v];
                }
                sum[v] += product[v] * factor[ORDER - 1][v];
            }
        };
        one(std::integral_constant<int, 0>{});
        one(std::integral_constant<int, 1>{});
        one(std::integral_constant<int, 2>{});
        one(std::integral_constant<int, 3>{});
    }
    const T total = sum_over_teams<T, V>(sum, exchange);
    sum_over_groups(
        output, total, partial + static_cast<size_t>(which) * groups * Layout::R, counters + which, group, groups,
        Layout::R, row0, n_rows
    );
}

// --------------------------------------------------------- the table turned --
/// Integers that make up a record: the offsets of the other factors, then the coefficient.
template <typename T, int ORDER> constexpr int record_size() { return ORDER - 1 + static_cast<int>(sizeof(T) / 4); }

__global__ __launch_bounds__(THREADS) void
count_kernel(int32_t* counts, const int32_t* __restrict__ P, int32_t n_pairs, int32_t nA, int32_t chunk) {
    extern __shared__ int32_t histogram[];
    for (int32_t f = threadIdx.x; f < nA; f += blockDim.x) {
        histogram[f] = 0;
    }
    __syncthreads();
    const int32_t begin = blockIdx.x * chunk, end = min(begin + chunk, n_pairs);
    for (int32_t p = begin + threadIdx.x; p < end; p += blockDim.x) {
        const int32_t f = P[p];
        if (in_bounds(f, nA)) {
            atomicAdd(histogram + f, 1);
        }
    }
    __syncthreads();
    for (int32_t f = threadIdx.x; f < nA; f += blockDim.x) {
        counts[static_cast<size_t>(blockIdx.x) * nA + f] = histogram[f];
    }
}

/// Stable counting sort of the pairs (monomial, factor) by feature, each pair
/// written as a record; the list of a feature starts at a multiple of four
/// records and is filled up with terms that are zero. A workgroup has
/// ROUNDS * 64 pairs per wavefront, in order; `counts` (count_kernel) says how
/// many of a feature the workgroups before it have. One workgroup needs none.
template <typename T, int ORDER, int ROUNDS>
__global__ __launch_bounds__(THREADS) void records_kernel(
    int32_t* lists,   // [nA + 1], in units of four records
    uint32_t* records,
    const int32_t* __restrict__ counts,
    const int32_t* __restrict__ P,
    const T* __restrict__ C,
    int32_t n_pairs,
    int32_t nA,
    int32_t stride, // bytes per feature of the tile the records are meant for
    int bits        // of a feature
) {
    constexpr int SIZE = record_size<T, ORDER>();
    extern __shared__ int32_t shared[];
    int32_t* start = shared;                                        // [nA]
    int32_t* of_wave = shared + nA;                                 // [16]
    uint16_t* seen = reinterpret_cast<uint16_t*>(of_wave + WAVES);  // [wavefronts][nA]
    const int waves = blockDim.x / WAVE;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    for (int32_t i = threadIdx.x; i < (waves * nA + 1) / 2; i += blockDim.x) {
        reinterpret_cast<uint32_t*>(seen)[i] = 0;
    }
    const int32_t first = (static_cast<int32_t>(blockIdx.x) * waves + wave) * (ROUNDS * WAVE) + lane;
    int32_t feature[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        const int32_t p = first + r * WAVE;
        feature[r] = p < n_pairs ? P[p] : -1;
    }
    __syncthreads();
    // how many pairs of the same feature come before, in this wavefront
    uint16_t* mine = seen + static_cast<size_t>(wave) * nA;
    uint32_t rank[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        const bool valid = in_bounds(feature[r], nA);
        uint64_t same = __ballot(valid);
        for (int b = 0; b < bits; b++) {
            const bool set = (feature[r] >> b & 1) != 0;
            const uint64_t with = __ballot(set);
            same &= set ? with : ~with;
        }
        const uint32_t before = __popcll(same & ((uint64_t(1) << lane) - 1));
        const uint32_t known = valid ? mine[feature[r]] : 0;
        rank[r] = known + before;
        __builtin_amdgcn_wave_barrier();
        if (valid && before == 0) {
            mine[feature[r]] = static_cast<uint16_t>(known + __popcll(same));
        }
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    // where every list starts: totals over all workgroups, rounded up to four, summed up
    int32_t carry = 0;
    for (int32_t base = 0; base < nA; base += blockDim.x) {
        const int32_t f = base + threadIdx.x;
        int32_t before = 0, total = 0;
        if (f < nA) {
            int32_t in_block = 0;
            for (int w = 0; w < waves; w++) {
                const int32_t of_this = seen[static_cast<size_t>(w) * nA + f];
                seen[static_cast<size_t>(w) * nA + f] = static_cast<uint16_t>(in_block);
                in_block += of_this;
            }
            if (gridDim.x == 1) {
                total = in_block;
            } else {
                int32_t after = 0;
#pragma unroll 8
                for (int32_t b = 0; b < static_cast<int32_t>(gridDim.x); b++) {
                    const int32_t count = counts[static_cast<size_t>(b) * nA + f];
                    before += b < static_cast<int32_t>(blockIdx.x) ? count : 0;
                    after += b < static_cast<int32_t>(blockIdx.x) ? 0 : count;
                }
                total = before + after;
            }
        }
        const int32_t quads = (total + TEAM - 1) / TEAM;
        int32_t scan = quads;
#pragma unroll
        for (int step = 1; step < WAVE; step <<= 1) {
            const int32_t other = __shfl_up(scan, step);
            scan += lane >= step ? other : 0;
        }
        if (lane == WAVE - 1) {
            of_wave[wave] = scan;
        }
        __syncthreads();
        int32_t ahead = carry;
        for (int w = 0; w < waves; w++) {
            const int32_t sum = of_wave[w];
            ahead += w < wave ? sum : 0;
            carry += sum;
        }
        if (f < nA) {
            const int32_t list = ahead + scan - quads;
            start[f] = list * TEAM + before;
            if (blockIdx.x == 0) {
                lists[f] = list;
                for (int32_t at = list * TEAM + total; at < (list + quads) * TEAM; at++) {
                    uint32_t* record = records + static_cast<size_t>(at) * SIZE;
#pragma unroll
                    for (int i = 0; i < SIZE; i++) {
                        record[i] = i < ORDER - 1 ? static_cast<uint32_t>(nA) * static_cast<uint32_t>(stride) : 0u;
                    }
                }
            }
        }
        __syncthreads();
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        lists[nA] = carry;
    }

#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        if (!in_bounds(feature[r], nA)) {
            continue;
        }
        const int32_t p = first + r * WAVE;
        const int32_t j = p / ORDER, k = p - j * ORDER;
        const int32_t at = start[feature[r]] + mine[feature[r]] + static_cast<int32_t>(rank[r]);
        uint32_t* record = records + static_cast<size_t>(at) * SIZE;
        const int32_t* factors = P + static_cast<size_t>(j) * ORDER;
#pragma unroll
        for (int i = 0; i < ORDER - 1; i++) {
            const uint32_t other = static_cast<uint32_t>(factors[i < k ? i : i + 1]);
            record[i] = min(other, static_cast<uint32_t>(nA)) * static_cast<uint32_t>(stride);
        }
        const T coefficient = C[j];
        __builtin_memcpy(record + ORDER - 1, &coefficient, sizeof(T));
    }
}

// ---------------------------------------------------------------- gradients --
/// A team per feature (or several, each with a share of its list: `log2_parts`)
/// adds up the terms of the feature's list for all rows of the tile. SECOND:
/// also their derivative along grad_grad_A, which is grad_A_2; the terms
/// themselves times grad_grad_A, over all features, are grad_grad_output.
template <typename T, int ORDER, int V, bool SECOND>
__global__ __launch_bounds__(THREADS) void gradient_kernel(
    T* grad_A,           // SECOND: grad_A_2, may be null
    T* grad_grad_output, // SECOND only, may be null
    T* partial,
    int32_t* counters,
    const T* __restrict__ grad_grad_A,
    const T* __restrict__ grad_output,
    const T* __restrict__ A,
    const int32_t* __restrict__ lists,
    const uint32_t* __restrict__ records,
    int32_t n_rows,
    int32_t nA,
    int32_t share, // features per workgroup
    int log2_parts,
    int32_t tiles,
    int32_t groups
) {
    constexpr int PARTS = SECOND ? 2 : 1;
    constexpr int OTHERS = ORDER - 1;
    constexpr int SIZE = record_size<T, ORDER>();
    using Layout = Tile<T, V, PARTS>;
    extern __shared__ __align__(16) char lds[];
    T* exchange = reinterpret_cast<T*>(lds);
    char* tile = lds + (SECOND ? WAVES * Layout::R * sizeof(T) : 0);
    int32_t which, group;
    if (!my_share(tiles, groups, which, group)) {
        return;
    }
    const int32_t row0 = which * Layout::R;
    const int team = threadIdx.x / TEAM, q = threadIdx.x & (TEAM - 1);
    const int part = team & ((1 << log2_parts) - 1);
    const int slot = team >> log2_parts;
    const int32_t begin = group * share, end = min(begin + share, nA);

    stage<T, V, PARTS>(tile, 0, A, row0, n_rows, nA);
    if constexpr (SECOND) {
        stage<T, V, PARTS>(tile, 1, grad_grad_A, row0, n_rows, nA);
    }
    const bool swap = (team & 1) != 0;
    T upstream[V];
#pragma unroll
    for (int v = 0; v < V; v++) {
        upstream[v] = grad_output[min(row0 + row_of<T, V>(q, v, swap), n_rows - 1)];
    }
    __syncthreads();

    const Layout values(tile, team, q);
    T along[V]; // SECOND: the share of grad_grad_output
#pragma unroll
    for (int v = 0; v < V; v++) {
        along[v] = T(0);
    }
    for (int32_t base = begin; base < end; base += TEAMS >> log2_parts) {
        const int32_t f = base + slot;
        const bool exists = f < end;
        const int32_t last = exists ? lists[f + 1] : 0;
        int32_t at = (exists ? lists[f] : 0) + part;
        T sum[V], derivative[V];
#pragma unroll
        for (int v = 0; v < V; v++) {
            sum[v] = T(0);
            derivative[v] = T(0);
        }
        uint32_t next[SIZE];
        auto fetch = [&](int32_t quad) { // (there are four spare records behind the last list)
            const uint32_t* record = records + (static_cast<size_t>(quad) * TEAM + q) * SIZE;
#pragma unroll
            for (int i = 0; i < SIZE; i++) {
                next[i] = record[i];
            }
        };
        if (at < last) {
            fetch(at);
        }
        for (; at < last; at += 1 << log2_parts) {
            Term<T, OTHERS> now;
#pragma unroll
            for (int i = 0; i < OTHERS; i++) {
                now.offset[i] = next[i];
            }
            __builtin_memcpy(&now.coefficient, next + OTHERS, sizeof(T));
            fetch(min(at + (1 << log2_parts), last));
            auto one = [&](auto lane) {
                constexpr int FROM = decltype(lane)::value;
                const T coefficient = from_lane<FROM>(now.coefficient);
                T factor[OTHERS > 0 ? OTHERS : 1][V];
                T tangent[OTHERS > 0 ? OTHERS : 1][V];
#pragma unroll
                for (int k = 0; k < OTHERS; k++) {
                    const uint32_t offset = from_lane<FROM>(now.offset[k]);
                    values.read(factor[k], offset);
                    if constexpr (SECOND) {
                        values.read(tangent[k], offset, 1);
                    }
                }
#pragma unroll
                for (int v = 0; v < V; v++) {
                    T product = coefficient;
                    T slope = T(0);
#pragma unroll
                    for (int k = 0; k < OTHERS; k++) {
                        if constexpr (SECOND) {
                            slope = slope * factor[k][v] + product * tangent[k][v];
                        }
                        if (k < OTHERS - 1) {
                            product *= factor[k][v];
                        }
                    }
                    if constexpr (OTHERS > 0) {
                        sum[v] += product * factor[OTHERS - 1][v];
                    } else {
                        sum[v] += product;
                    }
                    derivative[v] += slope;
                }
            };
            one(std::integral_constant<int, 0>{});
            one(std::integral_constant<int, 1>{});
            one(std::integral_constant<int, 2>{});
            one(std::integral_constant<int, 3>{});
        }
        if constexpr (SECOND) {
            T own[V];
            values.read(own, static_cast<uint32_t>(exists ? f : nA) * static_cast<uint32_t>(Layout::STRIDE), 1);
#pragma unroll
            for (int v = 0; v < V; v++) {
                along[v] += own[v] * sum[v];
            }
        }
        T result[V];
#pragma unroll
        for (int v = 0; v < V; v++) {
            result[v] = SECOND ? derivative[v] : sum[v];
        }
        if (log2_parts > 0) {
            // the teams of a feature lie in one wavefront; those that hold their halves the
            // other way round turn them
            if constexpr (V > 1 && V / chunk_values<T, V>() == 2) {
#pragma unroll
                for (int v = 0; v < V / 2; v++) {
                    const T low = result[v], high = result[v + V / 2];
                    result[v] = swap ? high : low;
                    result[v + V / 2] = swap ? low : high;
                }
            }
            for (int step = TEAM; step < TEAM << log2_parts; step <<= 1) {
#pragma unroll
                for (int v = 0; v < V; v++) {
                    result[v] += __shfl_xor(result[v], step);
                }
            }
        }
        if (exists && part == 0 && (!SECOND || grad_A != nullptr)) {
            const bool swapped = log2_parts == 0 && swap; // (part 0 is an even team otherwise)
#pragma unroll
            for (int v = 0; v < V; v++) {
                const int32_t row = row0 + row_of<T, V>(q, v, swapped);
                if (row < n_rows) {
                    grad_A[static_cast<size_t>(row) * nA + f] = upstream[v] * result[v];
                }
            }
        }
    }
    if constexpr (SECOND) {
        if (grad_grad_output != nullptr) {
            const T total = sum_over_teams<T, V>(along, exchange);
            sum_over_groups(
                grad_grad_output, total, partial + static_cast<size_t>(which) * groups * Layout::R, counters + which,
                group, groups, Layout::R, row0, n_rows
            );
        }
    }
}

// --------------------------------------------------------------------- host --
size_t tile_bytes(const Shape& s, size_t element_size, int values, int parts_per_feature) {
    return (static_cast<size_t>(s.nA) + 1) * parts_per_feature * TEAM * values * element_size;
}
size_t exchange_bytes(int values, size_t element_size) { return static_cast<size_t>(WAVES) * TEAM * values * element_size; }

struct Sort {
    int waves;
    int rounds;
    int32_t blocks;
    int32_t chunk;
};
Sort sort_of(const Shape& s) {
    const int32_t n_pairs = s.n_monomials * s.order;
    Sort sort;
    sort.waves = s.nA <= 3000 ? WAVES : 4; // (counters of every wavefront in LDS: 96 KB, 80 KB)
    // (many pairs in larger shares, because every workgroup adds up the counts of all others)
    sort.rounds = n_pairs <= (1 << 19) ? 4 : 16;
    sort.chunk = sort.waves * WAVE * sort.rounds;
    sort.blocks = static_cast<int32_t>(ceil_div(static_cast<size_t>(n_pairs), static_cast<size_t>(sort.chunk)));
    return sort;
}

/// Carves `bytes` of scratch memory; with no memory given, adds them up.
struct Carver {
    char* base;
    size_t used = 0;
    void* take(size_t bytes) {
        void* p = base + used;
        used += align256(bytes);
        return p;
    }
};
TurnedTable carve_table(const Shape& s, size_t element_size, Carver& carver) {
    const size_t n_pairs = static_cast<size_t>(s.n_monomials) * s.order;
    const Sort sort = sort_of(s);
    TurnedTable table;
    table.lists = static_cast<int32_t*>(carver.take((static_cast<size_t>(s.nA) + 1) * sizeof(int32_t)));
    table.counts = static_cast<int32_t*>(
        carver.take(sort.blocks > 1 ? static_cast<size_t>(sort.blocks) * s.nA * sizeof(int32_t) : 0)
    );
    table.records = static_cast<uint32_t*>(carver.take(
        (n_pairs + static_cast<size_t>(TEAM) * (s.nA + 1)) * (s.order - 1 + element_size / 4) * sizeof(uint32_t)
    ));
    return table;
}

struct Workspace {
    TurnedTable table;
    void* partial;
    size_t bytes;
};
Workspace carve(const Shape& s, const Plan& plan, size_t element_size, bool second, void* at) {
    Carver carver{static_cast<char*>(at)};
    Workspace w;
    w.table = carve_table(s, element_size, carver);
    w.partial = carver.take(
        second && plan.groups > 1 ? static_cast<size_t>(plan.tiles) * plan.groups * TEAM * plan.values * element_size : 0
    );
    w.bytes = carver.used;
    return w;
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
template <typename Body> void with_values(int values, Body&& body) {
    if (values == 1) {
        body(std::integral_constant<int, 1>{});
    } else if (values == 2) {
        body(std::integral_constant<int, 2>{});
    } else {
        body(std::integral_constant<int, MOST_VALUES>{});
    }
}

template <typename T, int ORDER>
void enqueue_table(const TurnedTable& w, const T* C, const int32_t* P, const Shape& s, int32_t stride, hipStream_t stream) {
    const int32_t n_pairs = s.n_monomials * s.order;
    const Sort sort = sort_of(s);
    if (sort.blocks > 1) {
        const size_t lds = static_cast<size_t>(s.nA) * sizeof(int32_t);
        count_kernel<<<sort.blocks, THREADS, lds, stream>>>(w.counts, P, n_pairs, s.nA, sort.chunk);
    }
    int bits = 1;
    while ((1 << bits) < s.nA) {
        bits++;
    }
    const size_t lds = (static_cast<size_t>(s.nA) + WAVES) * sizeof(int32_t) +
                       (static_cast<size_t>(sort.waves) * s.nA + 1) / 2 * sizeof(uint32_t);
    auto launch = [&](auto kernel) {
        allow_lds(kernel, lds);
        kernel<<<sort.blocks, sort.waves * WAVE, lds, stream>>>(
            w.lists, w.records, w.counts, P, C, n_pairs, s.nA, stride, bits
        );
    };
    if (sort.rounds == 4) {
        launch(records_kernel<T, ORDER, 4>);
    } else {
        launch(records_kernel<T, ORDER, 16>);
    }
}

template <typename T, bool SECOND>
void gradient(
    T* grad_A, T* grad_grad_output, const T* grad_grad_A, const T* grad_output, const T* A, const T* C,
    const int32_t* P, const Shape& s, const Plan& plan, void* workspace, int32_t* counters, hipStream_t stream
) {
    const Workspace w = carve(s, plan, sizeof(T), SECOND, workspace);
    const int32_t share = static_cast<int32_t>(ceil_div(static_cast<size_t>(s.nA), static_cast<size_t>(plan.groups)));
    with_order(s.order, [&](auto order) {
        constexpr int ORDER = decltype(order)::value;
        const int32_t stride = (SECOND ? 2 : 1) * TEAM * plan.values * static_cast<int32_t>(sizeof(T));
        enqueue_table<T, ORDER>(w.table, C, P, s, stride, stream);
        with_values(plan.values, [&](auto values) {
            auto kernel = gradient_kernel<T, ORDER, decltype(values)::value, SECOND>;
            allow_lds(kernel, plan.lds);
            MainKernelTimer timer(stream);
            kernel<<<blocks_of(plan), THREADS, plan.lds, stream>>>(
                grad_A, grad_grad_output, static_cast<T*>(w.partial), counters, grad_grad_A, grad_output, A, w.table.lists,
                w.table.records, s.n_rows, s.nA, share, plan.log2_parts, plan.tiles, plan.groups
            );
        });
    });
}

/// Values per lane and workgroups per tile, for `lds(values)` bytes of LDS and
/// at most `most_groups` workgroups per tile: the widest rows that still give
/// every compute unit a workgroup. (100 000 rows, 100 features, 2000 monomials
/// of order 4 in double, 4 / 2 / 1 values: forward 120 / 186 / 275 us, vjp 426 /
/// 488 / 505; 100 rows, 53 features, 28 794 monomials: vjp 40 / 32 / 31. Eight
/// values in float were never ahead of four.) Where the tile is read only a few
/// times, the time is in filling it: then as narrow as lets three workgroups
/// share a compute unit, one loading while another computes (17 886 rows, 1397
/// features, 314 monomials of order 3, forward, 4 / 2 values in float 33 / 24
/// us, 2 / 1 in double 66 / 52).
template <typename Bytes> Plan choose(const Shape& s, size_t most_groups, Bytes&& lds) {
    const size_t units = static_cast<size_t>(compute_units());
    const bool light = static_cast<size_t>(s.n_monomials) * s.order < 4 * static_cast<size_t>(s.nA);
    Plan plan;
    for (int values = MOST_VALUES; values >= 1; values >>= 1) {
        const size_t bytes = lds(values);
        if (bytes > LDS_LIMIT) {
            continue;
        }
        plan.values = values;
        plan.lds = bytes;
        plan.tiles = static_cast<int32_t>(ceil_div(static_cast<size_t>(s.n_rows), static_cast<size_t>(TEAM * values)));
        const size_t resident = units * (bytes <= LDS_LIMIT / 2 ? 2 : 1);
        plan.groups = static_cast<int32_t>(std::min(most_groups, std::max<size_t>(1, resident / plan.tiles)));
        if (plan.tiles * most_groups >= units && !(light && bytes > LDS_LIMIT / 3)) {
            break;
        }
    }
    return plan;
}

} // namespace

bool covered(const Shape& s) {
    return s.order >= 1 && s.order <= 6 && s.n_monomials > 0 && s.n_rows > 0 && s.nA > 0 &&
           static_cast<size_t>(s.n_monomials) * s.order < (size_t(1) << 28);
}

size_t table_bytes(const Shape& s, size_t element_size) {
    Carver carver{nullptr};
    carve_table(s, element_size, carver);
    return carver.used;
}

template <typename T>
TurnedTable turn_table(const T* C, const int32_t* P, const Shape& s, int32_t stride, void* workspace, hipStream_t stream) {
    Carver carver{static_cast<char*>(workspace)};
    const TurnedTable table = carve_table(s, sizeof(T), carver);
    with_order(s.order, [&](auto order) { enqueue_table<T, decltype(order)::value>(table, C, P, s, stride, stream); });
    return table;
}

Plan plan_forward(const Shape& s, size_t element_size) {
    Plan plan;
    if (!covered(s)) {
        return plan;
    }
    // (a share of fewer monomials than the workgroup has lanes leaves lanes idle)
    const size_t most_groups = std::max<size_t>(1, static_cast<size_t>(s.n_monomials) / THREADS);
    return choose(s, most_groups, [&](int values) {
        return tile_bytes(s, element_size, values, 1) + exchange_bytes(values, element_size);
    });
}

Plan plan_gradient(const Shape& s, size_t element_size, bool second) {
    if (!covered(s) || s.nA > MAX_FEATURES) {
        return Plan();
    }
    // (a feature can occupy sixteen teams: four features still occupy a quarter of a workgroup)
    const size_t most_groups = std::max<size_t>(1, static_cast<size_t>(s.nA) / 4);
    Plan plan = choose(s, most_groups, [&](int values) {
        return tile_bytes(s, element_size, values, second ? 2 : 1) +
               (second ? exchange_bytes(values, element_size) : 0);
    });
    if (plan.values > 0) {
        const size_t share = ceil_div(static_cast<size_t>(s.nA), static_cast<size_t>(plan.groups));
        plan.groups = static_cast<int32_t>(ceil_div(static_cast<size_t>(s.nA), share));
        while (plan.log2_parts < 4 && (share << (plan.log2_parts + 1)) <= TEAMS) {
            plan.log2_parts++;
        }
    }
    return plan;
}

size_t forward_bytes(const Shape& s, const Plan& plan, size_t element_size) {
    return plan.groups > 1 ? static_cast<size_t>(plan.tiles) * plan.groups * TEAM * plan.values * element_size : 0;
}
size_t gradient_bytes(const Shape& s, const Plan& plan, size_t element_size, bool second) {
    return carve(s, plan, element_size, second, nullptr).bytes;
}

template <typename T>
void forward(
    T* output, const T* A, const T* C, const int32_t* P, const Shape& s, const Plan& plan, void* workspace,
    int32_t* counters, hipStream_t stream
) {
    const int32_t share = static_cast<int32_t>(
        ceil_div(ceil_div(static_cast<size_t>(s.n_monomials), static_cast<size_t>(plan.groups)), TEAM) * TEAM
    );
    with_order(s.order, [&](auto order) {
        with_values(plan.values, [&](auto values) {
            auto kernel = forward_kernel<T, decltype(order)::value, decltype(values)::value>;
            allow_lds(kernel, plan.lds);
            MainKernelTimer timer(stream);
            kernel<<<blocks_of(plan), THREADS, plan.lds, stream>>>(
                output, static_cast<T*>(workspace), counters, A, C, P, s.n_rows, s.nA, s.n_monomials, share, plan.tiles,
                plan.groups
            );
        });
    });
}

template <typename T>
void vjp(
    T* grad_A, const T* grad_output, const T* A, const T* C, const int32_t* P, const Shape& s, const Plan& plan,
    void* workspace, hipStream_t stream
) {
    gradient<T, false>(grad_A, nullptr, nullptr, grad_output, A, C, P, s, plan, workspace, nullptr, stream);
}

template <typename T>
void vjp_vjp(
    T* grad_grad_output, T* grad_A_2, const T* grad_grad_A, const T* grad_output, const T* A, const T* C,
    const int32_t* P, const Shape& s, const Plan& plan, void* workspace, int32_t* counters, hipStream_t stream
) {
    gradient<T, true>(
        grad_A_2, grad_grad_output, grad_grad_A, grad_output, A, C, P, s, plan, workspace, counters, stream
    );
}

#define MOPS_INSTANTIATE(T)                                                                         \
    template void forward<T>(                                                                      \
        T*, const T*, const T*, const int32_t*, const Shape&, const Plan&, void*, int32_t*, hipStream_t \
    );                                                                                             \
    template void vjp<T>(                                                                          \
        T*, const T*, const T*, const T*, const int32_t*, const Shape&, const Plan&, void*, hipStream_t \
    );                                                                                             \
    template void vjp_vjp<T>(                                                                      \
        T*, T*, const T*, const T*, const T*, const T*, const int32_t*, const Shape&, const Plan&, void*, int32_t*, \
        hipStream_t                                                                                \
    );                                                                                             \
    template TurnedTable turn_table<T>(const T*, const int32_t*, const Shape&, int32_t, void*, hipStream_t);
MOPS_INSTANTIATE(float)
MOPS_INSTANTIATE(double)
#undef MOPS_INSTANTIATE

} // namespace hpe_tiles
} // namespace mops::amd
