#include "sender_buckets.hpp"

#include <algorithm>
#include <type_traits>

#include "runtime.hpp"
#include "sender_shares.hpp"
#include "wave_sort.hpp"

namespace mops::amd {

namespace {

// A stable counting sort of the edges by sender, in two levels where there are
// more senders than MOST_BUCKETS: into buckets of 2^shift consecutive senders,
// then every bucket by a workgroup of its own. Nothing is counted or placed by
// atomics on global memory (a returning atomic per edge, 1 000 000 of them over
// eight L2 caches, took 90 us): a workgroup counts its share of the edges, and
// the next launch finds out from all counts where its share of every bucket
// begins. Where edge and sender's place in its bucket fit into one word of 32 bits,
// the second level looks at nothing else, and both levels keep a lane's first items
// in registers from counting to placing. 1 000 000 edges over 33 000 senders: 35 us
// for the three launches (5, 15 and 15; 46 with two looks at everything), 400 000
// over 10 000: 27; what they wait for is one dependent load after the other.
constexpr int SORT_THREADS = 1024;
constexpr int32_t MOST_BUCKETS = 512;
constexpr int32_t SENDERS_AT_A_TIME = 4096;  // of the second level: counters in LDS

constexpr int HELD = 4;                      // positions a lane keeps from counting to placing
constexpr int32_t STAGED = 5120;             // edges of a bucket that are put in order in LDS

/// counts[workgroup][pitch]: how many in every bucket of the workgroup's share of the edges.
__global__ __launch_bounds__(SORT_THREADS) void count_buckets_kernel(
    int32_t* __restrict__ counts, const int32_t* __restrict__ senders, int32_t n_edges, int32_t n_nodes, int shift,
    int32_t pitch, int32_t share
) {
    __shared__ int32_t histogram[MOST_BUCKETS];
    for (int32_t b = threadIdx.x; b < pitch; b += SORT_THREADS) {
        histogram[b] = 0;
    }
    __syncthreads();
    const int32_t begin = blockIdx.x * share, end = begin + min(share, n_edges - begin);
    constexpr int AHEAD = 4;
    for (int32_t e = begin + threadIdx.x; e < end; e += AHEAD * SORT_THREADS) {
        int32_t sender[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            sender[u] = senders[min(e + u * SORT_THREADS, n_edges - 1)];
        }
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            if (e + u * SORT_THREADS < end && in_bounds(sender[u], n_nodes)) {
                atomicAdd(&histogram[sender[u] >> shift], 1);
            }
        }
    }
    __syncthreads();
    for (int32_t b = threadIdx.x; b < pitch; b += SORT_THREADS) {
        counts[static_cast<size_t>(blockIdx.x) * pitch + b] = histogram[b];
    }
}

/// The edges into their buckets, in ascending order. With one sender per bucket this is the result;
/// `offsets`: where every bucket begins, and where the last one ends. `pitch`: the buckets, rounded
/// up to a multiple of four.
/// LDS: counters[wavefronts][pitch], before[pitch], total[pitch], of_wave[wavefronts].
__global__ __launch_bounds__(SORT_THREADS) void fill_buckets_kernel(
    int32_t* __restrict__ sender_of_place, int32_t* __restrict__ edge_of_place, int32_t* __restrict__ offsets,
    const int32_t* __restrict__ counts, const int32_t* __restrict__ senders, int32_t n_edges, int32_t n_nodes, int shift,
    int32_t buckets, int32_t pitch, int bits, int32_t share, int packed_above
) {
    constexpr int WAVES = SORT_THREADS / WAVE;
    extern __shared__ int32_t shared[];
    int32_t* counters = shared;
    int32_t* before = counters + WAVES * pitch;
    int32_t* total = before + pitch;
    int32_t* of_wave = total + pitch;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const int32_t first = blockIdx.x * share, last = first + min(share, n_edges - first);
    const WaveShare mine(first, last, wave, WAVES);
    auto item_at = [&](int32_t e) {
        const int32_t sender = senders[e];
        return Item{in_bounds(sender, n_nodes) ? sender >> shift : -1, e, sender};
    };
    for (int32_t b = threadIdx.x; b < pitch; b += SORT_THREADS) {
        before[b] = 0;
        total[b] = 0;
    }
    const Held<HELD> held(mine, lane, item_at);
    count_keys<4>(held, counters, pitch, mine, wave, WAVES, lane, item_at);
    // what the workgroups before have of every bucket, and all of them: several threads per bucket
    // (of a single workgroup, the counts it has just made)
    const int32_t* all_counts = gridDim.x > 1 ? counts : counters;
    const int32_t rows = gridDim.x > 1 ? static_cast<int32_t>(gridDim.x) : WAVES;
    const int32_t mine_from = gridDim.x > 1 ? static_cast<int32_t>(blockIdx.x) : 0;
    const int32_t groups = pitch / 4; // (of four buckets)
    const int32_t group = static_cast<int32_t>(threadIdx.x) % groups;
    int4 ahead{0, 0, 0, 0}, all{0, 0, 0, 0};
#pragma unroll 8
    for (int32_t w = threadIdx.x / groups; w < rows; w += SORT_THREADS / groups) {
        const int4 count = reinterpret_cast<const int4*>(all_counts)[w * groups + group];
        const int32_t earlier = w < mine_from ? -1 : 0;
        ahead.x += count.x & earlier;
        ahead.y += count.y & earlier;
        ahead.z += count.z & earlier;
        ahead.w += count.w & earlier;
        all.x += count.x;
        all.y += count.y;
        all.z += count.z;
        all.w += count.w;
    }
    if (static_cast<int32_t>(threadIdx.x) < SORT_THREADS / groups * groups) {
        int32_t* to = before + 4 * group;
        atomicAdd(&to[0], ahead.x);
        atomicAdd(&to[1], ahead.y);
        atomicAdd(&to[2], ahead.z);
        atomicAdd(&to[3], ahead.w);
        to = total + 4 * group;
        atomicAdd(&to[0], all.x);
        atomicAdd(&to[1], all.y);
        atomicAdd(&to[2], all.z);
        atomicAdd(&to[3], all.w);
    }
    __syncthreads();
    const int32_t listed = scan_in_place<WAVES>(total, buckets, 0, of_wave);
    if (blockIdx.x == 0) {
        for (int32_t bucket = threadIdx.x; bucket < buckets; bucket += SORT_THREADS) {
            offsets[bucket] = total[bucket];
        }
        if (threadIdx.x == 0) {
            offsets[buckets] = listed;
        }
    }
    starts_of_waves<WAVES>(counters, pitch, [&](int32_t bucket) { return total[bucket] + before[bucket]; });
    // (two levels: the sender's place in its bucket beside the edge, where both go into one word)
    const int32_t of_bucket = (1 << shift) - 1;
    place_keys<4>(held, counters, pitch, bits, mine, wave, lane, item_at, [&](int32_t place, const Item& item) {
        edge_of_place[place] = packed_above < 32 ? item.edge | (item.sender & of_bucket) << packed_above : item.edge;
        if (sender_of_place != nullptr) {
            sender_of_place[place] = item.sender;
        }
    });
    // (places that no edge takes: as many as there are edges whose sender does not exist)
    for (int32_t place = max(first, listed) + static_cast<int32_t>(threadIdx.x); place < last; place += SORT_THREADS) {
        edge_of_place[place] = 0;
        if (sender_of_place != nullptr) {
            sender_of_place[place] = n_nodes;
        }
    }
}

/// A workgroup per bucket puts its edges in the order of their senders. The sender of a place's edge
/// is in the edge's word from bit `packed_above` on, or in `senders`. A bucket of up to `staged_room` edges
/// is put in order in LDS and written in whole lines (1 000 000 edges, 33 000 senders: 26.5 us with
/// two looks at `senders` by edge and stores of 64 words in 64 lines, 15.0 like this).
/// LDS: counters[wavefronts][at_a_time], start[at_a_time], of_wave[wavefronts], staged[staged_room].
template <int WAVES>
__global__ __launch_bounds__(WAVES* WAVE) void sort_buckets_kernel(
    int32_t* __restrict__ sender_of_place, int32_t* __restrict__ edge_of_place, int32_t* __restrict__ offsets,
    const int32_t* __restrict__ bucket_offsets, const int32_t* __restrict__ senders, const int32_t* __restrict__ edges,
    int packed_above, int32_t n_edges, int32_t n_nodes, int shift, int32_t at_a_time, int bits, int32_t staged_room
) {
    extern __shared__ int32_t shared[];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    int32_t* counters = shared;
    int32_t* start = counters + WAVES * at_a_time;
    int32_t* of_wave = start + at_a_time;
    int32_t* staged = of_wave + WAVES;
    const int32_t begin = bucket_offsets[blockIdx.x], end = bucket_offsets[blockIdx.x + 1];
    const WaveShare mine(begin, end, wave, WAVES);
    const int32_t node0 = static_cast<int32_t>(blockIdx.x) << shift;
    const int32_t nodes = min(1 << shift, n_nodes - node0);
    const bool packed = packed_above < 32;
    const bool in_lds = packed && end - begin <= staged_room && nodes <= at_a_time;
    const uint32_t edge_mask = packed ? (1u << packed_above) - 1 : ~0u;
    int32_t place0 = begin;
    for (int32_t base = 0; base < nodes; base += at_a_time) {
        const int32_t keys = min(at_a_time, nodes - base);
        auto item_at = [&](int32_t place) {
            const uint32_t word = static_cast<uint32_t>(edges[place]);
            const int32_t of_bucket =
                packed ? static_cast<int32_t>(word >> packed_above) : senders[place] - node0;
            const int32_t key = of_bucket - base;
            return Item{in_bounds(key, keys) ? key : -1, static_cast<int32_t>(word & edge_mask), node0 + of_bucket};
        };
        const Held<HELD> held(mine, lane, item_at);
        count_keys<4>(held, counters, keys, mine, wave, WAVES, lane, item_at);
        for (int32_t key = threadIdx.x; key < keys; key += blockDim.x) {
            int32_t sum = 0;
#pragma unroll
            for (int w = 0; w < WAVES; w++) {
                sum += counters[w * keys + key];
            }
            start[key] = sum;
        }
        __syncthreads();
        place0 = scan_in_place<WAVES>(start, keys, place0, of_wave);
        for (int32_t key = threadIdx.x; key < keys; key += blockDim.x) {
            offsets[node0 + base + key] = start[key];
        }
        starts_of_waves<WAVES>(counters, keys, [&](int32_t key) { return start[key]; });
        place_keys<4>(held, counters, keys, bits, mine, wave, lane, item_at, [&](int32_t place, const Item& item) {
            if (in_lds) {
                staged[place - begin] = item.edge | item.key << packed_above;
            } else {
                edge_of_place[place] = item.edge;
                if (sender_of_place != nullptr) {
                    sender_of_place[place] = item.sender;
                }
            }
        });
        __syncthreads();
    }
    if (in_lds) {
        for (int32_t place = begin + static_cast<int32_t>(threadIdx.x); place < end; place += WAVES * WAVE) {
            const uint32_t word = static_cast<uint32_t>(staged[place - begin]);
            edge_of_place[place] = static_cast<int32_t>(word & edge_mask);
            if (sender_of_place != nullptr) {
                sender_of_place[place] = node0 + static_cast<int32_t>(word >> packed_above);
            }
        }
    }
    if (blockIdx.x == gridDim.x - 1) {
        if (threadIdx.x == 0) {
            offsets[n_nodes] = end;
        }
        for (int32_t place = end + static_cast<int32_t>(threadIdx.x); place < n_edges; place += blockDim.x) {
            edge_of_place[place] = 0;
            if (sender_of_place != nullptr) {
                sender_of_place[place] = n_nodes;
            }
        }
    }
}

constexpr int SPLIT_THREADS = 512;

__global__ __launch_bounds__(SPLIT_THREADS) void
split_shares_kernel(const Shares to, const SharePlan plan, const int32_t* __restrict__ senders) {
    extern __shared__ int32_t lds[];
    split_share<SPLIT_THREADS>(lds, to, plan, senders, blockIdx.x);
}

// Sparse graphs: one launch of list_in_slots_block (sender_buckets.hpp), four
// wavefronts per workgroup.
constexpr int SLOT_THREADS = 4 * WAVE;

__global__ __launch_bounds__(SLOT_THREADS) void list_in_slots_kernel(
    int32_t* __restrict__ slots, int32_t* __restrict__ counts, const int32_t* __restrict__ senders,
    int32_t n_edges, int32_t n_nodes, bool aligned
) {
    __shared__ SlotLists lists;
    list_in_slots_block<SLOT_THREADS>(lists, slots, counts, senders, n_edges, n_nodes, aligned, blockIdx.x);
}

// Sparse graphs, by arrival: one thread per edge.
constexpr int ARRIVAL_THREADS = 4 * WAVE;

__global__ __launch_bounds__(ARRIVAL_THREADS) void list_by_arrival_kernel(
    const SenderArrivals lists, const int32_t* __restrict__ senders, int32_t n_edges, int32_t n_nodes
) {
    const int32_t edge = static_cast<int32_t>(blockIdx.x) * ARRIVAL_THREADS + static_cast<int32_t>(threadIdx.x);
    if (edge < n_edges) {
        list_arrival(lists, n_nodes, senders[edge], edge);
    }
}

__global__ __launch_bounds__(ARRIVAL_THREADS) void clear_counters_kernel(int32_t* __restrict__ counters, size_t count) {
    const size_t at = static_cast<size_t>(blockIdx.x) * ARRIVAL_THREADS + threadIdx.x;
    if (at < count) {
        counters[at] = 0;
    }
}

} // namespace

size_t sender_slots_bytes(int32_t n_nodes) {
    return align256(static_cast<size_t>(n_nodes) * SLOT_CAPACITY * 4) +
           align256(static_cast<size_t>(n_nodes) * SLOT_PARTS * 4);
}

SenderSlots sender_slots_in(void* workspace, int32_t n_nodes) {
    int32_t* slots = static_cast<int32_t*>(workspace);
    int32_t* counts = reinterpret_cast<int32_t*>(
        static_cast<char*>(workspace) + align256(static_cast<size_t>(n_nodes) * SLOT_CAPACITY * 4)
    );
    return SenderSlots{slots, counts};
}

unsigned sender_slots_blocks(int32_t n_nodes) {
    return static_cast<unsigned>(ceil_div(static_cast<size_t>(std::max(n_nodes, 0)), SLOT_SENDERS)) * SLOT_PARTS;
}

SenderSlots list_edges_in_slots(
    const int32_t* senders, int32_t n_edges, int32_t n_nodes, void* workspace, hipStream_t stream
) {
    const SenderSlots slots = sender_slots_in(workspace, n_nodes);
    if (n_nodes > 0) {
        const bool aligned = reinterpret_cast<uintptr_t>(senders) % 16 == 0;
        list_in_slots_kernel<<<sender_slots_blocks(n_nodes), SLOT_THREADS, 0, stream>>>(
            const_cast<int32_t*>(slots.edges), const_cast<int32_t*>(slots.counts), senders, n_edges, n_nodes, aligned
        );
        MOPS_HIP_CHECK(hipGetLastError());
    }
    return slots;
}

SenderArrivals list_edges_by_arrival(
    const int32_t* senders, int32_t n_edges, int32_t n_nodes, int32_t copies, void* workspace, int32_t* counts,
    hipStream_t stream
) {
    const SenderArrivals lists{static_cast<int32_t*>(workspace), counts, copies};
    if (n_nodes > 0 && n_edges > 0) {
        const unsigned blocks = static_cast<unsigned>(ceil_div(static_cast<size_t>(n_edges), ARRIVAL_THREADS));
        list_by_arrival_kernel<<<blocks, ARRIVAL_THREADS, 0, stream>>>(lists, senders, n_edges, n_nodes);
        MOPS_HIP_CHECK(hipGetLastError());
    }
    return lists;
}

void clear_counters(int32_t* counters, size_t count, hipStream_t stream) {
    if (count > 0) {
        const unsigned blocks = static_cast<unsigned>(ceil_div(count, ARRIVAL_THREADS));
        clear_counters_kernel<<<blocks, ARRIVAL_THREADS, 0, stream>>>(counters, count);
        MOPS_HIP_CHECK(hipGetLastError());
    }
}

namespace {

struct SortPlan {
    int shift;       // senders per bucket: 2^shift
    int32_t buckets, pitch;
    int32_t share;   // edges per workgroup of the first level
    int32_t shares;
    int packed_above; // two levels: bits below the sender's place in its bucket, 32: not in one word
};
int bits_for(int32_t values) {
    int bits = 0;
    while ((int64_t(1) << bits) < values) {
        bits++;
    }
    return bits;
}
SortPlan sort_plan(int32_t n_nodes, int32_t n_edges) {
    SortPlan plan;
    plan.shift = 0;
    while ((n_nodes - 1) >> plan.shift >= MOST_BUCKETS) {
        plan.shift++;
    }
    plan.buckets = ((n_nodes - 1) >> plan.shift) + 1;
    plan.pitch = (plan.buckets + 3) / 4 * 4;
    const size_t each = ceil_div(static_cast<size_t>(n_edges), static_cast<size_t>(SORT_THREADS) * MOST_SHARES);
    plan.share = static_cast<int32_t>(each) * SORT_THREADS;
    plan.shares = static_cast<int32_t>(ceil_div(static_cast<size_t>(n_edges), static_cast<size_t>(plan.share)));
    const int edge_bits = bits_for(n_edges);
    plan.packed_above = plan.shift > 0 && edge_bits + plan.shift <= 32 ? edge_bits : 32;
    return plan;
}
} // namespace

bool plan_shares(SharePlan& plan, int32_t n_nodes, int32_t n_edges, int32_t buckets) {
    if (n_nodes < 1 || n_edges < 1 || buckets < 1 || buckets > n_nodes || buckets > MOST_SHARE_BUCKETS) {
        return false;
    }
    plan.n_edges = n_edges;
    plan.n_nodes = n_nodes;
    const size_t each = ceil_div(static_cast<size_t>(n_edges), static_cast<size_t>(MOST_SHARES) * SHARE_STEP);
    plan.share = static_cast<int32_t>(each) * SHARE_STEP;
    plan.shares = static_cast<int32_t>(ceil_div(static_cast<size_t>(n_edges), static_cast<size_t>(plan.share)));
    plan.buckets = buckets;
    plan.multiplier = 0;
    plan.senders_each = 0;
    plan.per_bucket = 1;
    if (buckets < n_nodes) {
        plan.multiplier = static_cast<uint32_t>((static_cast<uint64_t>(buckets) << 32) / static_cast<uint64_t>(n_nodes));
        plan.senders_each = 4294967296.0 / plan.multiplier;
        plan.per_bucket = static_cast<int32_t>((uint64_t(1) << 32) / plan.multiplier + 1);
    }
    plan.sender_bits = bits_for(plan.per_bucket);
    return each * SHARE_STEP <= MOST_SHARE_EDGES && plan.per_bucket <= MOST_PER_BUCKET &&
           bits_for(n_edges) + plan.sender_bits <= 32 &&
           static_cast<int64_t>(n_edges) <= static_cast<int64_t>(buckets) * BUCKET_EDGES / 4 * 3;
}

size_t shares_bytes(const SharePlan& plan, int32_t copies) {
    return align256(static_cast<size_t>(plan.shares) * plan.share * 4) +
           align256(static_cast<size_t>(plan.buckets) * plan.shares * 4) +
           static_cast<size_t>(copies) * plan.n_edges * 4;
}

Shares shares_in(void* workspace, const SharePlan& plan) {
    char* at = static_cast<char*>(workspace);
    Shares shares;
    shares.words = reinterpret_cast<uint32_t*>(at);
    at += align256(static_cast<size_t>(plan.shares) * plan.share * 4);
    shares.starts = reinterpret_cast<uint32_t*>(at);
    at += align256(static_cast<size_t>(plan.buckets) * plan.shares * 4);
    shares.lists = reinterpret_cast<int32_t*>(at);
    return shares;
}

void split_shares(const Shares& to, const SharePlan& plan, const int32_t* senders, hipStream_t stream) {
    const size_t lds = static_cast<size_t>(split_lds<SPLIT_THREADS>(plan.buckets)) * sizeof(int32_t);
    split_shares_kernel<<<plan.shares, SPLIT_THREADS, lds, stream>>>(to, plan, senders);
    MOPS_HIP_CHECK(hipGetLastError());
}

size_t edges_by_sender_bytes(int32_t n_nodes, int32_t n_edges, bool with_senders) {
    if (n_nodes < 1) {
        return 0;
    }
    const bool senders_in_buckets = n_edges > 0 && sort_plan(n_nodes, n_edges).packed_above == 32;
    return align256((static_cast<size_t>(n_nodes) + 1) * 4) + align256((MOST_BUCKETS + 1) * 4) +
           (2 + with_senders + senders_in_buckets) * align256(static_cast<size_t>(n_edges) * 4);
}

EdgesBySender order_edges_by_sender(
    const int32_t* senders, int32_t n_edges, int32_t n_nodes, bool with_senders, void* workspace, hipStream_t stream
) {
    if (n_nodes < 1) {
        return EdgesBySender{nullptr, nullptr, nullptr};
    }
    char* at = static_cast<char*>(workspace);
    auto take = [&](size_t integers) {
        int32_t* p = reinterpret_cast<int32_t*>(at);
        at += align256(integers * 4);
        return p;
    };
    int32_t* offsets = take(static_cast<size_t>(n_nodes) + 1);
    int32_t* bucket_offsets = take(MOST_BUCKETS + 1);
    int32_t* edge = take(static_cast<size_t>(n_edges));
    int32_t* edge_in_buckets = take(static_cast<size_t>(n_edges));
    int32_t* sender = with_senders ? take(static_cast<size_t>(n_edges)) : nullptr;
    if (n_edges < 1) {
        clear_counters(offsets, static_cast<size_t>(n_nodes) + 1, stream);
        return EdgesBySender{sender, edge, offsets};
    }
    const SortPlan plan = sort_plan(n_nodes, n_edges);
    const bool two_levels = plan.shift > 0;
    int32_t* sender_in_buckets = plan.packed_above == 32 ? take(static_cast<size_t>(n_edges)) : nullptr;
    // The counts of several shares lie where nothing is written by the launch that reads them. They
    // fit: a share is 1024 edges or more, and there are 512 buckets at most.
    int32_t* counts = two_levels ? edge : edge_in_buckets;
    if (plan.shares > 1) {
        count_buckets_kernel<<<plan.shares, SORT_THREADS, 0, stream>>>(
            counts, senders, n_edges, n_nodes, plan.shift, plan.pitch, plan.share
        );
    }
    constexpr int WAVES = SORT_THREADS / WAVE;
    const size_t lds = (static_cast<size_t>(WAVES + 2) * plan.pitch + WAVES) * sizeof(int32_t);
    fill_buckets_kernel<<<plan.shares, SORT_THREADS, lds, stream>>>(
        two_levels ? sender_in_buckets : sender, two_levels ? edge_in_buckets : edge,
        two_levels ? bucket_offsets : offsets, counts, senders, n_edges, n_nodes, plan.shift, plan.buckets,
        plan.pitch, bits_for(plan.buckets), plan.share, plan.packed_above
    );
    if (two_levels) {
        const int32_t at_a_time = std::min(int32_t(1) << plan.shift, SENDERS_AT_A_TIME);
        // (the counters of all wavefronts within 64 KB)
        auto sort = [&](auto with_waves) {
            constexpr int WAVES = decltype(with_waves)::value;
            const int32_t room = WAVES >= 4 ? STAGED : 0;
            const size_t sort_lds = (static_cast<size_t>(WAVES + 1) * at_a_time + WAVES + room) * sizeof(int32_t);
            sort_buckets_kernel<WAVES><<<plan.buckets, WAVES * WAVE, sort_lds, stream>>>(
                sender, edge, offsets, bucket_offsets, sender_in_buckets, edge_in_buckets,
                plan.packed_above, n_edges, n_nodes, plan.shift, at_a_time, bits_for(at_a_time), room
            );
        };
        // (within 64 KB: the counters of all wavefronts, and the edges of a bucket where there is room)
        if (at_a_time <= 512) {
            sort(std::integral_constant<int, 16>{});
        } else if (at_a_time <= 1024) {
            sort(std::integral_constant<int, 8>{});
        } else if (at_a_time <= 2048) {
            sort(std::integral_constant<int, 4>{});
        } else {
            sort(std::integral_constant<int, 2>{});
        }
    }
    MOPS_HIP_CHECK(hipGetLastError());
    return EdgesBySender{sender, edge, offsets};
}

} // namespace mops::amd
