// The steps of a stable counting sort by a workgroup, without atomics on global memory: every
// wavefront counts a consecutive share of the positions, and places the items of its share in
// their order by the lanes of the same key (see sender_buckets.hip, sender_shares.hpp).
#ifndef MOPS_AMD_WAVE_SORT_HPP
#define MOPS_AMD_WAVE_SORT_HPP

#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "device_common.hpp"

namespace mops::amd {

// BATCH, below: positions beyond the held ones that a lane asks for at once.

/// What lies at a position: an edge, its sender, and what it is sorted by (negative: it is not).
struct Item {
    int32_t key, edge, sender;
};

/// The lanes of a wavefront with the same key, and how many of them are below this one.
struct Ranked {
    uint64_t same;
    uint32_t before;
};
__device__ __forceinline__ Ranked rank_in_wave(int32_t key, bool valid, int bits, int lane) {
    uint64_t same = __ballot(valid);
    for (int b = 0; b < bits; b++) {
        const bool set = (key >> b & 1) != 0;
        const uint64_t with = __ballot(set);
        same &= set ? with : ~with;
    }
    return Ranked{same, static_cast<uint32_t>(__popcll(same & ((uint64_t(1) << lane) - 1)))};
}

/// A wavefront's share [begin, end) of the positions a workgroup has.
struct WaveShare {
    int32_t begin, end;
    __device__ __forceinline__ WaveShare(int32_t first, int32_t last, int wave, int waves) {
        const int32_t each = ((last - first + waves - 1) / waves + WAVE - 1) / WAVE * WAVE;
        begin = min(first + wave * each, last);
        end = min(begin + each, last);
    }
};

/// The first N items of a lane: those of most shares all told, so that they are read once.
template <int N> struct Held {
    Item item[N];

    template <typename ItemAt> __device__ __forceinline__ Held(const WaveShare& share, int lane, ItemAt&& item_at) {
#pragma unroll
        for (int u = 0; u < N; u++) {
            item[u] = item_at(max(min(share.begin + u * WAVE + lane, share.end - 1), 0));
        }
    }
};
template <> struct Held<0> {
    Item item[1];
};

/// counters[wavefront][key] := how many of the wavefront's items have the key.
template <int BATCH, int HELD, typename ItemAt>
__device__ __forceinline__ void count_keys(
    const Held<HELD>& held, int32_t* counters, int32_t keys, const WaveShare& share, int wave, int waves, int lane,
    ItemAt&& item_at
) {
    for (int32_t i = threadIdx.x; i < waves * keys; i += blockDim.x) {
        counters[i] = 0;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < HELD; u++) {
        if (share.begin + u * WAVE + lane < share.end && held.item[u].key >= 0) {
            atomicAdd(&counters[wave * keys + held.item[u].key], 1);
        }
    }
#pragma unroll 1
    for (int32_t at = share.begin + HELD * WAVE + lane; at - lane < share.end; at += BATCH * WAVE) {
        int32_t key[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            key[u] = item_at(min(at + u * WAVE, share.end - 1)).key;
        }
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            if (at + u * WAVE < share.end && key[u] >= 0) {
                atomicAdd(&counters[wave * keys + key[u]], 1);
            }
        }
    }
    __syncthreads();
}

/// put(place, item) for every item that has a key, items of one key in ascending places:
/// counters[wavefront][key] is the place of the wavefront's first one.
template <int BATCH, int HELD, typename ItemAt, typename Put>
__device__ __forceinline__ void place_keys(
    const Held<HELD>& held, int32_t* counters, int32_t keys, int bits, const WaveShare& share, int wave, int lane,
    ItemAt&& item_at, Put&& put
) {
    int32_t* mine = counters + static_cast<size_t>(wave) * keys;
    auto place_one = [&](const Item& item, int32_t at) {
        const bool valid = at < share.end && item.key >= 0;
        const Ranked ranked = rank_in_wave(item.key, valid, bits, lane);
        const int32_t place = valid ? mine[item.key] + static_cast<int32_t>(ranked.before) : 0;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid && ranked.before == 0) {
            mine[item.key] += __popcll(ranked.same);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (valid) {
            put(place, item);
        }
    };
#pragma unroll
    for (int u = 0; u < HELD; u++) {
        if (share.begin + u * WAVE < share.end) { // (uniform)
            place_one(held.item[u], share.begin + u * WAVE + lane);
        }
    }
#pragma unroll 1
    for (int32_t at = share.begin + HELD * WAVE + lane; at - lane < share.end; at += BATCH * WAVE) {
        Item item[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            item[u] = item_at(min(at + u * WAVE, share.end - 1));
        }
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            place_one(item[u], at + u * WAVE);
        }
    }
}

/// The same for many keys, of which few are named twice among 64 items: the places come from atomics on the counters,
/// which lanes with the same key are given in no particular order; those are found by their places and put in
/// theirs. BATCH x 64 items wait for LDS together. (1 000 000 senders in shares of 4096 over 1024 buckets, two
/// wavefronts each, beside the edges' gradients of OPSAW: 4 us of the launch instead of 9.)
template <int BATCH, typename ItemAt, typename Put>
__device__ __forceinline__ void place_rare_keys(
    int32_t* counters, int32_t keys, const WaveShare& share, int wave, int lane, ItemAt&& item_at, Put&& put
) {
    int32_t* mine = counters + static_cast<size_t>(wave) * keys;
#pragma unroll 1
    for (int32_t at = share.begin + lane; at - lane < share.end; at += BATCH * WAVE) {
        Item item[BATCH];
        int32_t place[BATCH], given[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            item[u] = item_at(min(at + u * WAVE, share.end - 1));
            item[u].key = at + u * WAVE < share.end ? item[u].key : -1;
        }
#pragma unroll
        for (int u = 0; u < BATCH; u++) { // (LDS operations of one wavefront happen in program order)
            place[u] = given[u] = 0;
            if (item[u].key >= 0) {
                place[u] = __hip_atomic_load(&mine[item[u].key], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                given[u] = atomicAdd(&mine[item[u].key], 1);
            }
        }
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            uint64_t others = __ballot(given[u] != place[u]);
            while (others != 0) { // (uniform)
                const int32_t key = __builtin_amdgcn_readlane(item[u].key, __builtin_ctzll(others));
                const uint64_t same = __ballot(item[u].key == key);
                const int32_t before = __popcll(same & ((uint64_t(1) << lane) - 1));
                place[u] += item[u].key == key ? before : 0;
                others &= ~same;
            }
            if (item[u].key >= 0) {
                put(place[u], item[u]);
            }
        }
    }
}

/// Turns counters[wavefront][key] into the place of the wavefront's first of each key:
/// start_of(key) and what the wavefronts before have. All threads.
template <int WAVES, typename StartOf>
__device__ __forceinline__ void starts_of_waves(int32_t* counters, int32_t keys, StartOf&& start_of) {
    for (int32_t key = threadIdx.x; key < keys; key += blockDim.x) {
        int32_t here[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            here[w] = counters[w * keys + key];
        }
        int32_t place = start_of(key);
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            counters[w * keys + key] = place;
            place += here[w];
        }
    }
    __syncthreads();
}

/// values[0 .. n) := `first` + the sum of those before; returns `first` + the sum of all. All
/// threads; `of_wave`: an integer per wavefront.
template <int WAVES>
__device__ __forceinline__ int32_t scan_in_place(int32_t* values, int32_t n, int32_t first, int32_t* of_wave) {
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    int32_t carry = first;
    for (int32_t base = 0; base < n; base += blockDim.x) {
        const int32_t i = base + threadIdx.x;
        const int32_t value = i < n ? values[i] : 0;
        int32_t sum = value;
#pragma unroll
        for (int step = 1; step < WAVE; step <<= 1) {
            const int32_t other = __shfl_up(sum, step);
            sum += lane >= step ? other : 0;
        }
        if (lane == WAVE - 1) {
            of_wave[wave] = sum;
        }
        __syncthreads();
        int32_t ahead = carry;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            ahead += w < wave ? of_wave[w] : 0;
            carry += of_wave[w];
        }
        if (i < n) {
            values[i] = ahead + sum - value;
        }
        __syncthreads();
    }
    return carry;
}

} // namespace mops::amd

#endif
