// The per-edge gradients of OPSA / OPSAW for gfx950:
//
//   U[e, l]      = sum_k A[e, k] * gO[node, k, l]
//   grad_B[e, l] = U[e, l] * W[sender, l],   edge_W[e, l] = U[e, l] * B[e, l]
//   grad_A[e, k] = sum_l (B[e, l] * W[sender, l]) * gO[node, k, l]
//
// (without W: 1). A wavefront walks over the edges of a range, up to 16 of one
// node at a time: two products on the matrix cores, whose right operand is the
// node's block of grad_output. The rows of an edge have odd lengths and no
// alignment in general, so nothing is loaded in the layout of an operand: the 16
// rows of A and of B are one piece of memory each, rows of W are put together 64
// elements at a time, all of it goes through LDS (rows of odd length there: no
// bank meets more than two lanes), and so do the gradients on their way out. The
// block of a node is brought once for all its edges. Everything a tile needs is
// asked for while the one before is worked on, and nothing is left out by a
// branch between the asking and the waiting: what is not wanted, or not there, is
// asked of a tensor of no bytes.
//
// What bounds it on many edges is memory: 1 000 000 edges over 33 000 nodes, 13 x 32,
// f32, OPSAW, 134 us for 701 MB at the memory side of L2 (5.2 TB/s; the tensors have
// 551 MB; 155 us with the operands' layout loaded as it is), OPSA with 13 x 33 202 -> 121 us, 31 x 45 506 -> 202. Few tiles per
// wavefront (below 30 000 to 400 000 edges, by shape) are the other kernel's: this one
// has a start of some microseconds and as many wavefronts as are resident at most.
#include "opsa_edges.hpp"

#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "mfma.hpp"
#include "runtime.hpp"
#include "sasaw_table.hpp"
#include "sender_buckets.hpp"

namespace mops::amd::opsa_edges {
namespace {

using sasaw::BufferOf;
using sasaw::unless;
using sasaw::wave_sync;

constexpr int WAVES = 2; // per workgroup; they do not wait for each other
constexpr int THREADS = WAVES * WAVE;

/// Places of a wavefront's LDS, in elements. Rows are padded with zeros to whole
/// steps of four of the products, and to an odd length.
struct Places {
    int32_t pitch_A, pitch_L;
    int32_t B, W, G, all;
};
template <int KT, int LT> __host__ __device__ Places places_of(int32_t K, int32_t L, bool weighted) {
    Places p;
    p.pitch_A = (K + 3) / 4 * 4 | 1;
    p.pitch_L = (L + 3) / 4 * 4 | 1;
    p.B = 16 * p.pitch_A;
    p.W = p.B + 16 * p.pitch_L;
    p.G = p.W + (weighted ? 16 * p.pitch_L : 0);
    p.all = p.G + (K + 3) / 4 * 4 * p.pitch_L;
    return p;
}

template <typename T> struct Arguments {
    Tensors<T> t;
    int32_t ranges, range_edges;
    uint32_t reciprocal_K, reciprocal_L; // ceil(2^20 / .): rows of elements below 2048, in 24-bit products
    int32_t* slots;
    int32_t* slot_counts;
    int32_t list_blocks; // (none, but slots: every edge takes a place of its sender, see SenderArrivals)
    bool aligned_senders;
    SharePlan plan; // (no shares: the senders are not split)
    Shares shares;
    int32_t late, less; // the first `late` ranges have `less` edges less than the others
};

/// A tensor's rows first .. first + n, as elements 64 t + lane of one piece; n = 0: nothing.
template <typename T>
__device__ __forceinline__ BufferOf<T> piece_of(const T* tensor, int64_t first, int32_t n, int32_t length) {
    BufferOf<T> piece;
    piece.set(tensor + first * length, static_cast<uint32_t>(n * length) * static_cast<uint32_t>(sizeof(T)));
    return piece;
}

template <typename T, int KT, int LT, bool WEIGHTED>
__global__ __launch_bounds__(THREADS) void edge_kernel(const Arguments<T> p) {
    using M = Mfma<T>;
    constexpr uint32_t ES = sizeof(T);
    constexpr int LOADS_A = 4 * KT, LOADS_B = 4 * LT, LOADS_G = 4 * KT * LT;
    extern __shared__ __align__(16) char lds[];
    if constexpr (WEIGHTED) {
        if (static_cast<int32_t>(blockIdx.x) < p.list_blocks) {
            list_in_slots_block<THREADS>(
                *reinterpret_cast<SlotLists*>(lds), p.slots, p.slot_counts, p.t.senders, p.t.n_edges, p.t.n_nodes,
                p.aligned_senders, blockIdx.x
            );
            return;
        }
    }
    if constexpr (WEIGHTED) {
        // (a share of the senders first; the ranges of these workgroups are the shorter for it)
        if (static_cast<int32_t>(blockIdx.x) < p.plan.shares) {
            split_share<THREADS>(reinterpret_cast<int32_t*>(lds), p.shares, p.plan, p.t.senders, blockIdx.x);
            __syncthreads();
        }
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE); // (uniform, and known to be)
    const int lane = threadIdx.x & (WAVE - 1), i = lane & 15, q = lane >> 4;
    const int32_t range = (static_cast<int32_t>(blockIdx.x) - p.list_blocks) * WAVES + wave;
    if (range >= p.ranges) {
        return;
    }
    const int32_t K = p.t.K, L = p.t.L;
    const Places at = places_of<KT, LT>(K, L, WEIGHTED);
    T* const base = reinterpret_cast<T*>(lds) + wave * at.all;
    T *const a_tile = base, *const b_tile = base + at.B, *const w_tile = base + at.W, *const g_block = base + at.G;
    for (int32_t k = lane; k < at.all; k += WAVE) {
        base[k] = T(0); // (the padding stays so)
    }
    wave_sync();

    auto begin_of = [&](int32_t which) {
        const int64_t at = static_cast<int64_t>(which) * p.range_edges - p.less * min(which, p.late);
        return static_cast<int32_t>(at < p.t.n_edges ? at : p.t.n_edges);
    };
    const int32_t begin = begin_of(range), end = begin_of(range + 1);
    const bool want_A = p.t.grad_A != nullptr, want_U = p.t.grad_B != nullptr || (WEIGHTED && p.t.edge_W != nullptr);
    BufferOf<T> W;
    W.set(p.t.W, WEIGHTED ? static_cast<uint32_t>(p.t.n_nodes) * static_cast<uint32_t>(L) * ES : 0);

    // positions `first` .. of the indices, one per lane
    struct Window {
        int32_t receiver, sender;
    };
    auto window_at = [&](int32_t first) {
        const int32_t position = min(first + lane, p.t.n_edges - 1);
        return Window{p.t.receivers[position], WEIGHTED ? p.t.senders[position] : 0};
    };
    // the edges of one node from `from` places into the window at `first`: up to 16
    auto run = [&](const Window& w, int32_t first, int32_t from) {
        const int32_t node = __builtin_amdgcn_readlane(w.receiver, from);
        const unsigned long long others = __ballot(first + lane >= end || w.receiver != node) >> from;
        return others == 0 ? 16 : min(__ffsll(static_cast<long long>(others)) - 1, 16);
    };

    // The lane, of which the compiler knows nothing: places in LDS are computed where they are used, and
    // not kept in dozens of registers from one use to the next.
    auto fresh = [&] {
        uint32_t unknown = lane;
        asm volatile("" : "+v"(unknown));
        return unknown;
    };
    struct Rows {
        T a[LOADS_A], b[LOADS_B], w[WEIGHTED ? LOADS_B : 1];
    };
    // the places in their senders' lists of the n edges at `first`, which is `from` places into the window
    const bool arrivals = WEIGHTED && p.list_blocks == 0 && p.slots != nullptr;
    struct Arrival {
        int32_t sender, place;
    };
    auto arrive = [&](const Window& window, int32_t from, int32_t n) {
        Arrival arrival{0, SLOT_CAPACITY};
        if (arrivals) {
            arrival.sender = __builtin_amdgcn_ds_bpermute((from + lane) << 2, window.sender);
            if (lane < n && in_bounds(arrival.sender, p.t.n_nodes)) {
                arrival.place = atomicAdd(&p.slot_counts[arrival.sender], 1);
            }
        }
        return arrival;
    };
    // rows of the n edges at `first`, which is `from` places into the window
    auto ask_rows = [&](Rows& rows, const Window& window, int32_t first, int32_t from, int32_t n) {
        const BufferOf<T> A = piece_of(p.t.A, first, n, K), B = piece_of(p.t.B, first, n, L);
        const uint32_t lane = fresh();
#pragma unroll
        for (int t = 0; t < LOADS_A; t++) {
            rows.a[t] = A.load((t * WAVE + lane) * ES, 0);
        }
#pragma unroll
        for (int t = 0; t < LOADS_B; t++) {
            rows.b[t] = B.load((t * WAVE + lane) * ES, 0);
        }
        if constexpr (WEIGHTED) {
#pragma unroll
            for (int t = 0; t < LOADS_B; t++) {
                const uint32_t x = t * WAVE + lane, row = __umul24(x, p.reciprocal_L) >> 20;
                const int32_t sender = __builtin_amdgcn_ds_bpermute((from + row) << 2, window.sender);
                const uint32_t element = x + (static_cast<uint32_t>(sender) - row) * static_cast<uint32_t>(L);
                rows.w[t] = W.load(
                    element * ES | unless(static_cast<int32_t>(row) < n && in_bounds(sender, p.t.n_nodes)), 0
                );
            }
        }
    };
    auto place = [&](uint32_t x, uint32_t reciprocal, int32_t length, int32_t pitch) {
        return x + __umul24(__umul24(x, reciprocal) >> 20, static_cast<uint32_t>(pitch - length));
    };

    Window window = window_at(begin);
    int32_t first = begin, n = run(window, begin, 0), block = -1;
    Rows rows;
    T g[LOADS_G];
    Arrival arrival = arrive(window, 0, n);
    ask_rows(rows, window, first, 0, n);
    auto ask_block = [&](int32_t node) {
        // (a node that does not exist: zeros)
        const bool exists = in_bounds(node, p.t.n_nodes);
        const BufferOf<T> G = piece_of(p.t.grad_output, exists ? static_cast<int64_t>(node) * K : 0, exists ? K : 0, L);
        const uint32_t lane = fresh();
#pragma unroll
        for (int t = 0; t < LOADS_G; t++) {
            g[t] = G.load((t * WAVE + lane) * ES, 0);
        }
    };
    int32_t node = __builtin_amdgcn_readlane(window.receiver, 0);
    ask_block(node);
    while (true) {
        // the tile to LDS
        const uint32_t lane_in = fresh();
#pragma unroll
        for (int t = 0; t < LOADS_A; t++) {
            const uint32_t x = t * WAVE + lane_in;
            if (static_cast<int32_t>(x) < 16 * K) {
                a_tile[place(x, p.reciprocal_K, K, at.pitch_A)] = rows.a[t];
            }
        }
#pragma unroll
        for (int t = 0; t < LOADS_B; t++) {
            const uint32_t x = t * WAVE + lane_in;
            if (static_cast<int32_t>(x) < 16 * L) {
                const uint32_t to = place(x, p.reciprocal_L, L, at.pitch_L);
                b_tile[to] = rows.b[t];
                if constexpr (WEIGHTED) {
                    w_tile[to] = rows.w[t];
                }
            }
        }
        if (node != block) {
            block = node;
#pragma unroll
            for (int t = 0; t < LOADS_G; t++) {
                const uint32_t x = t * WAVE + lane_in;
                if (static_cast<int32_t>(x) < K * L) {
                    g_block[place(x, p.reciprocal_L, L, at.pitch_L)] = g[t];
                }
            }
        }
        if (arrival.place < SLOT_CAPACITY) {
            p.slots[static_cast<size_t>(arrival.sender) * SLOT_CAPACITY + arrival.place] = first + lane;
        }
        wave_sync();

        // the next one
        const int32_t next_first = first + n;
        const bool more = next_first < end;
        const int32_t next_n = more ? run(window, first, n) : 0;
        const int32_t next_node = __builtin_amdgcn_readlane(window.receiver, n);
        arrival = arrive(window, n, next_n);
        ask_rows(rows, window, next_first, n, next_n);
        const Window next_window = window_at(next_first);
        if (more && next_node != block) {
            ask_block(next_node);
        }
        __builtin_amdgcn_sched_barrier(0);

        typename M::Acc sum_A[KT], U[LT];
#pragma unroll
        for (int t = 0; t < KT; t++) {
            sum_A[t] = M::zero();
        }
#pragma unroll
        for (int t = 0; t < LT; t++) {
            U[t] = M::zero();
        }
        if (want_A) {
            const T *const b_row = b_tile + i * at.pitch_L + q, *const w_row = w_tile + i * at.pitch_L + q;
            const T* g_row[KT];
#pragma unroll
            for (int t = 0; t < KT; t++) {
                g_row[t] = g_block + min(16 * t + i, K - 1) * at.pitch_L + q;
            }
#pragma unroll
            for (int s = 0; s < 4 * LT; s++) {
                if (4 * s < L) { // (uniform)
                    const T left = WEIGHTED ? b_row[4 * s] * w_row[4 * s] : b_row[4 * s];
#pragma unroll
                    for (int t = 0; t < KT; t++) {
                        sum_A[t] = M::mma(left, g_row[t][4 * s], sum_A[t]);
                    }
                }
            }
        }
        if (want_U) {
            const T* const a_row = a_tile + i * at.pitch_A + q;
            const T* g_column[LT];
#pragma unroll
            for (int t = 0; t < LT; t++) {
                g_column[t] = g_block + q * at.pitch_L + min(16 * t + i, L - 1);
            }
#pragma unroll
            for (int s = 0; s < 4 * KT; s++) {
                if (4 * s < K) { // (uniform)
                    const T left = a_row[4 * s];
#pragma unroll
                    for (int t = 0; t < LT; t++) {
                        U[t] = M::mma(left, g_column[t][4 * s * at.pitch_L], U[t]);
                    }
                }
            }
        }
        wave_sync();
        // the gradients take the places of what they are made from
#pragma unroll
        for (int t = 0; t < LT; t++) {
            const int32_t l = 16 * t + i;
            if (l < L) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int32_t e = M::row(lane, r) * at.pitch_L + l;
                    if constexpr (WEIGHTED) {
                        const T b = b_tile[e], w = w_tile[e];
                        w_tile[e] = U[t][r] * b;
                        b_tile[e] = U[t][r] * w;
                    } else {
                        b_tile[e] = U[t][r];
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < KT; t++) {
            const int32_t k = 16 * t + i;
            if (k < K) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    a_tile[M::row(lane, r) * at.pitch_A + k] = sum_A[t][r];
                }
            }
        }
        wave_sync();
        const uint32_t lane_out = fresh(), last = at.all - 1; // (elements that nothing takes are read from there)
        const BufferOf<T> to_A = piece_of(p.t.grad_A, first, want_A ? n : 0, K);
        const BufferOf<T> to_B = piece_of(p.t.grad_B, first, p.t.grad_B != nullptr ? n : 0, L);
#pragma unroll
        for (int t = 0; t < LOADS_A; t++) {
            const uint32_t x = t * WAVE + lane_out;
            to_A.store(a_tile[min(place(x, p.reciprocal_K, K, at.pitch_A), last)], x * ES, 0);
        }
#pragma unroll
        for (int t = 0; t < LOADS_B; t++) {
            const uint32_t x = t * WAVE + lane_out;
            to_B.store(a_tile[min(at.B + place(x, p.reciprocal_L, L, at.pitch_L), last)], x * ES, 0);
        }
        if constexpr (WEIGHTED) {
            const BufferOf<T> to_W = piece_of(p.t.edge_W, first, p.t.edge_W != nullptr ? n : 0, L);
#pragma unroll
            for (int t = 0; t < LOADS_B; t++) {
                const uint32_t x = t * WAVE + lane_out;
                to_W.store(a_tile[min(at.W + place(x, p.reciprocal_L, L, at.pitch_L), last)], x * ES, 0);
            }
        }
        if (!more) {
            break;
        }
        wave_sync();
        first = next_first;
        n = next_n;
        node = next_node;
        window = next_window;
    }
}

template <typename T, int KT, int LT, bool WEIGHTED>
void launch_with(
    const Tensors<T>& t, int32_t* slots, int32_t* slot_counts, unsigned list_blocks, const SharePlan* plan,
    const Shares& shares, hipStream_t stream
) {
    Arguments<T> p{};
    p.t = t;
    if (plan != nullptr) {
        p.plan = *plan;
        p.shares = shares;
    }
    p.slots = slots;
    p.slot_counts = slot_counts;
    p.list_blocks = static_cast<int32_t>(list_blocks);
    p.aligned_senders = reinterpret_cast<uintptr_t>(t.senders) % 16 == 0;
    auto reciprocal = [](int32_t n) { return ((1u << 20) + static_cast<uint32_t>(n) - 1) / static_cast<uint32_t>(n); };
    p.reciprocal_K = reciprocal(t.K);
    p.reciprocal_L = reciprocal(t.L);
    const Places at = places_of<KT, LT>(t.K, t.L, WEIGHTED);
    // (readers of the last row may look up to 64 elements beyond it)
    size_t lds = (static_cast<size_t>(WAVES) * at.all + 64 * LT + 64) * sizeof(T);
    if (list_blocks > 0) {
        lds = std::max(lds, sizeof(SlotLists));
    }
    if (plan != nullptr) {
        lds = std::max(lds, split_lds<THREADS>(plan->buckets) * sizeof(int32_t));
    }
    auto kernel = edge_kernel<T, KT, LT, WEIGHTED>;
    if (lds > 64 * 1024) {
        MOPS_HIP_CHECK(hipFuncSetAttribute(
            reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)
        ));
    }
    const int64_t resident = static_cast<int64_t>(compute_units()) * WAVES *
                             std::max<int64_t>(1, std::min<int64_t>(8, static_cast<int64_t>(160 * 1024 / lds)));
    const int64_t tiles = (static_cast<int64_t>(t.n_edges) + 15) / 16;
    const int64_t per_range = (tiles + resident - 1) / resident;
    p.range_edges = static_cast<int32_t>(std::min<int64_t>(16 * per_range, 1 << 30));
    if (plan != nullptr) {
        p.late = static_cast<int32_t>(std::min<int64_t>(plan->shares * WAVES, resident));
        // (splitting 1024 edges takes as long as what moves some 15 000 bytes of a wavefront's range)
        const int64_t edge_bytes = static_cast<int64_t>(2 * t.K + 5 * t.L) * static_cast<int64_t>(sizeof(T));
        p.less = static_cast<int32_t>(std::min(15000 * (plan->share / 1024) / edge_bytes, t.n_edges / resident / 2));
        p.range_edges = static_cast<int32_t>((t.n_edges + static_cast<int64_t>(p.late) * p.less + resident - 1) / resident);
    }
    p.ranges = static_cast<int32_t>(
        (static_cast<int64_t>(t.n_edges) + static_cast<int64_t>(p.late) * p.less + p.range_edges - 1) / p.range_edges
    );
    const unsigned blocks =
        std::max(list_blocks + static_cast<unsigned>((p.ranges + WAVES - 1) / WAVES), static_cast<unsigned>(p.plan.shares));
    kernel<<<blocks, THREADS, lds, stream>>>(p);
    MOPS_HIP_CHECK(hipGetLastError());
}

} // namespace

bool covers(int32_t n_nodes, int32_t K, int32_t L, size_t element_size) {
    return n_nodes > 0 && K > 0 && K <= 32 && L > 0 && L <= 64 &&
           static_cast<uint64_t>(n_nodes) * static_cast<uint64_t>(L) * element_size < (uint64_t(1) << 32);
}

template <typename T>
void launch(
    const Tensors<T>& t, int32_t* slots, int32_t* slot_counts, unsigned list_blocks, const SharePlan* plan,
    const Shares& shares, hipStream_t stream
) {
    auto with_columns = [&](auto kt, auto lt) {
        constexpr int KT = decltype(kt)::value, LT = decltype(lt)::value;
        if (t.W != nullptr) {
            launch_with<T, KT, LT, true>(t, slots, slot_counts, list_blocks, plan, shares, stream);
        } else {
            launch_with<T, KT, LT, false>(t, slots, slot_counts, list_blocks, plan, shares, stream);
        }
    };
    auto with_rows = [&](auto kt) {
        if (t.L <= 16) {
            with_columns(kt, std::integral_constant<int, 1>{});
        } else if (t.L <= 32) {
            with_columns(kt, std::integral_constant<int, 2>{});
        } else if (t.L <= 48) {
            with_columns(kt, std::integral_constant<int, 3>{});
        } else {
            with_columns(kt, std::integral_constant<int, 4>{});
        }
    };
    if (t.K <= 16) {
        with_rows(std::integral_constant<int, 1>{});
    } else {
        with_rows(std::integral_constant<int, 2>{});
    }
}

template void launch<float>(const Tensors<float>&, int32_t*, int32_t*, unsigned, const SharePlan*, const Shares&, hipStream_t);
template void launch<double>(const Tensors<double>&, int32_t*, int32_t*, unsigned, const SharePlan*, const Shares&, hipStream_t);

} // namespace mops::amd::opsa_edges
