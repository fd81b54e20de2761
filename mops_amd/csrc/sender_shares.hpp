// Edges grouped by an UNSORTED index without a launch of its own in series: a
// stable counting sort whose first half rides along with a kernel that does not
// need the lists, and whose second half is done by the kernel that does.
//
//   split_share    a workgroup puts its share of the edges into the order of
//                  their buckets (per_bucket consecutive senders each) and
//                  writes down where every bucket begins in it. It needs
//                  nothing from other workgroups: some workgroups of a launch
//                  with other work do it (or split_shares_kernel).
//   gather_bucket  a workgroup that is going to work on a bucket's senders
//                  fetches the bucket's edges from all shares, in order, and
//                  sorts them by sender in LDS.
//
// What both wait for is chains of loads and the fetching of instructions that run
// once, so that neither is worth a launch. SASAW, 9 components, 32 columns, whole vjp,
// f32 / f64, us, against a launch that lists the edges in places of their senders
// (60 000 edges; 8.4 us in series) or three for order_edges_by_sender (36 us of
// 1 000 000): 60 000 edges of 2000 nodes 51.5 -> 45.8 / 65 -> 60; 60 000 of 1000
// 67 -> 51 (f32); 200 000 of 6600 117 -> 99.6 / 186 -> 164; 1 000 000 of 33 000 478 ->
// 446 / 855 -> 818. The places of a bucket of up to eight senders counted in
// registers, with two barriers instead of nine, was 2 us slower: more instructions
// to fetch. Alone (grad_W and nothing else) the split is a launch of 5 to 14 us.
#ifndef MOPS_AMD_SENDER_SHARES_HPP
#define MOPS_AMD_SENDER_SHARES_HPP

#include <cstdint>

#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "wave_sort.hpp"

namespace mops::amd {

constexpr int32_t MOST_SHARES = 256;
constexpr int32_t SHARE_STEP = 1024;        // edges of a share: a multiple of this
constexpr int32_t MOST_SHARE_EDGES = 32768; // (places in a share take 16 bits)
constexpr int32_t MOST_SHARE_BUCKETS = 1024; // counters in LDS, of every wavefront
/// Edges of a bucket that fit into LDS. Larger ones (of a few senders with many more
/// edges than the others: on average buckets are at most three quarters of it) are sorted in global memory.
constexpr int32_t BUCKET_EDGES = 2048;
constexpr int32_t MOST_PER_BUCKET = 512;

struct SharePlan {
    int32_t n_edges, n_nodes;
    int32_t share, shares;        // edges of a share (the last one may have fewer), and how many shares
    int32_t buckets, per_bucket;  // of senders, and how many senders at most
    uint32_t multiplier;          // floor(2^32 buckets / n_nodes); 0: a bucket per sender
    double senders_each;          // 2^32 / multiplier
    int sender_bits; // of a sender's place in its bucket

    __device__ __forceinline__ int32_t bucket_of(int32_t sender) const {
        return multiplier == 0 ? sender : static_cast<int32_t>(__umulhi(static_cast<uint32_t>(sender), multiplier));
    }
    /// The first sender of a bucket: the smallest whose product with the multiplier reaches bucket * 2^32.
    __device__ __forceinline__ int32_t first_of(int32_t bucket) const {
        const int32_t about = static_cast<int32_t>(bucket * senders_each); // (or one less)
        return multiplier == 0 ? bucket : min(about + (bucket_of(about) < bucket ? 1 : 0), n_nodes);
    }
};

/// The plan with so many buckets; false: a graph for order_edges_by_sender.
bool plan_shares(SharePlan& plan, int32_t n_nodes, int32_t n_edges, int32_t buckets);

/// Consecutive numbers to the workgroups of one die (which get every eighth workgroup): what consecutive buckets
/// have of a share lies on the same lines, eight buckets to a line of 128 bytes if they have four edges each.
/// Workgroups below `count` only; of a launch of swizzled_blocks(count).
constexpr int32_t DIES = 8;
__device__ __forceinline__ int32_t swizzled(int32_t block, int32_t count) {
    return block % DIES * ((count + DIES - 1) / DIES) + block / DIES;
}
inline int32_t swizzled_blocks(int32_t count) { return (count + DIES - 1) / DIES * DIES; }

/// What the first half leaves behind.
struct Shares {
    uint32_t* words;  // [shares][share] edge in the share | lower half of its sender << 16, by bucket
    uint32_t* starts; // [shares][buckets] first of the bucket's places in the share | how many << 16
    int32_t* lists;   // [copies][n_edges] for buckets that do not fit into LDS
};
/// Bytes of scratch memory: `copies` workgroups gather the same bucket.
size_t shares_bytes(const SharePlan& plan, int32_t copies);
Shares shares_in(void* workspace, const SharePlan& plan);
/// Enqueue the first half as a launch of its own.
void split_shares(const Shares& to, const SharePlan& plan, const int32_t* senders, hipStream_t stream);

/// Integers of LDS that split_share takes.
template <int THREADS> __host__ __device__ constexpr int32_t split_lds(int32_t buckets) {
    return THREADS / WAVE * buckets + THREADS + THREADS / WAVE;
}

/// All threads of a workgroup of THREADS.
template <int THREADS>
__device__ __forceinline__ void
split_share(int32_t* lds, const Shares& to, const SharePlan& plan, const int32_t* __restrict__ senders, int32_t which) {
    constexpr int WAVES = THREADS / WAVE, BATCH = SHARE_STEP / THREADS < 8 ? SHARE_STEP / THREADS : 8;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    int32_t* counters = lds;
    int32_t* of_thread = counters + WAVES * plan.buckets;
    int32_t* of_wave = of_thread + THREADS;
    const int32_t first = which * plan.share, last = first + min(plan.share, plan.n_edges - first);
    const WaveShare mine(first, last, wave, WAVES);
    auto item_at = [&](int32_t e) {
        const int32_t sender = senders[e];
        const int32_t bucket = plan.bucket_of(sender);
        return Item{in_bounds(sender, plan.n_nodes) ? bucket : -1, e, sender};
    };
    count_keys<BATCH>(Held<0>{}, counters, plan.buckets, mine, wave, WAVES, lane, item_at);
    // every thread has as many consecutive buckets
    const int32_t each = (plan.buckets + THREADS - 1) / THREADS;
    const int32_t begin = min(static_cast<int32_t>(threadIdx.x) * each, plan.buckets), end = min(begin + each, plan.buckets);
    int32_t sum = 0;
    for (int32_t bucket = begin; bucket < end; bucket++) {
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            sum += counters[w * plan.buckets + bucket];
        }
    }
    of_thread[threadIdx.x] = sum;
    __syncthreads();
    scan_in_place<WAVES>(of_thread, THREADS, 0, of_wave);
    uint32_t* const starts = to.starts + static_cast<size_t>(which) * plan.buckets;
    int32_t place = of_thread[threadIdx.x];
    for (int32_t bucket = begin; bucket < end; bucket++) {
        const int32_t start = place;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            const int32_t here = counters[w * plan.buckets + bucket];
            counters[w * plan.buckets + bucket] = place;
            place += here;
        }
        starts[bucket] = static_cast<uint32_t>(start | (place - start) << 16);
    }
    __syncthreads();
    uint32_t* const words = to.words + first;
    place_rare_keys<BATCH>(counters, plan.buckets, mine, wave, lane, item_at, [&](int32_t place, const Item& item) {
        words[place] = static_cast<uint32_t>(item.edge - first) | static_cast<uint32_t>(item.sender) << 16;
    });
}

/// A bucket's edges, ascending for every sender; of its sender k places offsets[k] to offsets[k + 1].
struct BucketEdges {
    const int32_t* list;      // in LDS, if they fit
    const int32_t* in_memory; // if not
    const int32_t* offsets;   // in LDS
    int32_t* counter;         // in LDS
    int32_t n;
    bool fits;
};

/// Integers of LDS that gather_bucket takes: what stays (the last is a counter that starts at zero), and what is
/// needed for a while only.
__host__ __device__ constexpr int32_t bucket_lds(int32_t per_bucket) { return BUCKET_EDGES + per_bucket + 2; }
template <int THREADS> __host__ __device__ constexpr int32_t gather_lds(int32_t per_bucket) {
    return BUCKET_EDGES + MOST_SHARES + 2 * (THREADS / WAVE) + (THREADS / WAVE) * per_bucket;
}

/// What a thread has of a bucket: its edges in the share of the thread's number. Asked for in two steps, so that
/// a workgroup can do other things while the first, and then the second is on its way.
struct BucketFetch {
    static constexpr int HELD = 4;
    const uint32_t* words;
    int32_t start, count;
    uint32_t word[HELD]; // the first of them

    __device__ __forceinline__ BucketFetch(const Shares& from, const SharePlan& plan, int32_t bucket) {
        const int32_t share = min(static_cast<int32_t>(threadIdx.x), plan.shares - 1);
        const uint32_t found = from.starts[static_cast<size_t>(share) * plan.buckets + bucket];
        start = static_cast<int32_t>(threadIdx.x) < plan.shares ? static_cast<int32_t>(found & 0xffff) : 0;
        count = static_cast<int32_t>(threadIdx.x) < plan.shares ? static_cast<int32_t>(found >> 16) : 0;
        words = from.words + static_cast<size_t>(share) * plan.share;
    }
    __device__ __forceinline__ void ask() {
        words += start;
#pragma unroll
        for (int u = 0; u < HELD; u++) {
            word[u] = count > 0 ? words[min(u, count - 1)] : 0;
        }
    }
};

/// All threads of a workgroup of THREADS, which is in step afterwards. `copy`: of those that gather the bucket.
template <int THREADS>
__device__ __forceinline__ BucketEdges gather_bucket(
    int32_t* kept, int32_t* temporary, const BucketFetch& mine, const Shares& from, const SharePlan& plan, int32_t bucket,
    int32_t copy
) {
    static_assert(THREADS >= MOST_SHARES, "a thread per share");
    constexpr int WAVES = THREADS / WAVE;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const int32_t thread = threadIdx.x, node0 = plan.first_of(bucket);
    // (senders of a bucket are less than 2^16 apart)
    auto key_of = [&](uint32_t word) { return (word >> 16) - static_cast<uint32_t>(node0) & 0xffff; };
    int32_t* list = kept;
    int32_t* offsets = list + BUCKET_EDGES;
    uint32_t* raw = reinterpret_cast<uint32_t*>(temporary); // edge | the sender's place above it, by share
    int32_t* before = temporary + BUCKET_EDGES;              // [MOST_SHARES] of the bucket's edges
    int32_t* of_wave = before + MOST_SHARES;                 // [2 * WAVES]
    int32_t* counters = of_wave + 2 * WAVES;                 // [WAVES][per_bucket]
    const int32_t count = mine.count;
    int32_t* const counter = offsets + plan.per_bucket + 1;
    if (thread == 0) {
        *counter = 0;
        list[0] = 0; // (an edge that exists, for who looks at a place before the count; an edge takes it if there is one)
    }
    // how many the shares before have of this bucket, and all shares of the buckets before
    int32_t sum = count, earlier = mine.start;
#pragma unroll
    for (int step = 1; step < WAVE; step <<= 1) {
        const int32_t other = __shfl_up(sum, step), start_of_other = __shfl_xor(earlier, step);
        sum += lane >= step ? other : 0;
        earlier += start_of_other;
    }
    if (lane == WAVE - 1) {
        of_wave[wave] = sum;
        of_wave[WAVES + wave] = earlier;
    }
    __syncthreads();
    int32_t ahead = sum - count, n = 0, base = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        ahead += w < wave ? of_wave[w] : 0;
        n += of_wave[w];
        base += of_wave[WAVES + w];
    }
    n = __builtin_amdgcn_readfirstlane(n);
    base = __builtin_amdgcn_readfirstlane(base);
    if (thread < MOST_SHARES) {
        before[thread] = ahead;
    }
    const bool fits = n <= BUCKET_EDGES, sorted = plan.per_bucket == 1; // (uniform)
    int32_t* const in_memory = from.lists + static_cast<size_t>(copy) * plan.n_edges + base;
    const int above = 32 - plan.sender_bits;
    if (fits) {
        uint32_t* const to = sorted ? reinterpret_cast<uint32_t*>(list) : raw;
        auto put = [&](int32_t i, uint32_t word) {
            const uint32_t edge = static_cast<uint32_t>(thread * plan.share) + (word & 0xffff);
            if (i < count) {
                to[ahead + i] = sorted ? edge : edge | key_of(word) << above;
            }
        };
        constexpr int AHEAD = BucketFetch::HELD;
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            put(u, mine.word[u]);
        }
        for (int32_t i = AHEAD; i < count; i += AHEAD) {
            uint32_t word[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; u++) {
                word[u] = mine.words[min(i + u, count - 1)];
            }
#pragma unroll
            for (int u = 0; u < AHEAD; u++) {
                put(i + u, word[u]);
            }
        }
    }
    if (sorted && thread < 2) {
        offsets[thread] = thread * n;
    }
    __syncthreads();
    // by sender: a counting sort, of the places in LDS or of those in memory
    const WaveShare share(0, n, wave, WAVES);
    auto sort = [&](auto&& item_at, auto&& put) {
        // (nothing unrolled: what runs once is bound by the fetching of its instructions, too)
        const Held<0> none{};
        count_keys<1>(none, counters, plan.per_bucket, share, wave, WAVES, lane, item_at);
        for (int32_t key = thread; key < plan.per_bucket; key += THREADS) {
            int32_t all = 0;
#pragma unroll
            for (int w = 0; w < WAVES; w++) {
                all += counters[w * plan.per_bucket + key];
            }
            offsets[key] = all;
        }
        __syncthreads();
        scan_in_place<WAVES>(offsets, plan.per_bucket, 0, of_wave);
        starts_of_waves<WAVES>(counters, plan.per_bucket, [&](int32_t key) { return offsets[key]; });
        if (thread == 0) {
            offsets[plan.per_bucket] = n;
        }
        place_keys<1>(none, counters, plan.per_bucket, plan.sender_bits, share, wave, lane, item_at, put);
        __syncthreads();
    };
    if (!fits) {
        sort(
            [&](int32_t place) { // (the last share that has no more edges before it than this)
                int32_t which = 0;
#pragma unroll
                for (int step = MOST_SHARES / 2; step > 0; step /= 2) {
                    which += before[which + step] <= place ? step : 0;
                }
                const uint32_t of_share = from.starts[static_cast<size_t>(which) * plan.buckets + bucket] & 0xffff;
                const uint32_t word =
                    from.words[static_cast<size_t>(which) * plan.share + of_share + (place - before[which])];
                return Item{static_cast<int32_t>(key_of(word)), which * plan.share + static_cast<int32_t>(word & 0xffff), 0};
            },
            [&](int32_t place, const Item& item) { in_memory[place] = item.edge; }
        );
    } else if (!sorted) {
        sort(
            [&](int32_t place) {
                const uint32_t word = raw[place];
                return Item{static_cast<int32_t>(word >> above), static_cast<int32_t>(word & ((1u << above) - 1)), 0};
            },
            [&](int32_t place, const Item& item) { list[place] = item.edge; }
        );
    }
    return BucketEdges{list, in_memory, offsets, counter, n, fits};
}

} // namespace mops::amd

#endif
