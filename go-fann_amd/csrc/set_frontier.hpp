// set_frontier.hpp -- the beam's frontier as a set held in registers.
//
// The reference keeps the frontier in a symmetric min-max heap
// (include/smmh2.h) and scans its array for the next entry
// (pickup_next_unused_from_native_frontier, backend_pq.cu:844-892).  While
// the keys differ, neither the entry that pop_max takes nor the one that the
// scan takes depends on the array's order: they are the greatest of all
// entries and the least of the unused ones.  So the keys live in registers,
// position 64 j + lane in register j of that lane, and an admission to a full
// frontier overwrites the greatest key and finds the new one by a wave
// maximum, without the heap's chain of dependent LDS reads.
//
// Where keys are equal the array's order does decide, and it is a function of
// the admitted keys in admission order alone (used marks and payloads never
// move an entry).  That sequence is logged, and the heap is brought up to
// date from the log -- by the wave heap operations of device_common.hpp,
// from where it stood last -- only when an answer depends on it:
//   * two unused entries share the least key: the one of lower heap index is
//     next;
//   * an entry of the greatest key leaves while others have that key: which
//     one is left open (top_gone counts them).  It settles itself when the
//     rest of them leave too, which is what mostly happens; if one of them is
//     about to be picked, the heap says which are left.
// Of 380 admissions of a u8 route at Q = 72 (integer distances, so keys meet
// often) the heap saw 84, of 1,100 of an f16 route at Q = 416 it saw 15.  One u8
// route takes 248 us, with the heap 369; which launches take it, and why not
// all, is said where they are chosen (exact_route.hip).
// A NaN key has no place in such an order: from the first one on (eager) every
// admission goes through the heap as well.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>

#include "device_common.hpp"
#include "gofann_internal.hpp"

namespace gofann {

constexpr uint32_t kSetSlack = 16;  // positions past Q for entries whose leaving is open

// LDS bytes of a SplitHeap for a beam of q (Q + 2 slots).
__host__ __device__ inline uint32_t split_heap_bytes(int q)
{
    return (static_cast<uint32_t>(q) + 2u) * 6u;
}
__device__ __forceinline__ SplitHeap split_heap(unsigned char* lds, int q)
{
    float* f = reinterpret_cast<float*>(lds);
    return SplitHeap{f, reinterpret_cast<uint16_t*>(f + q + 2)};
}

// Positions of a beam of q in r registers a lane.
__host__ __device__ inline uint32_t set_capacity(int q, int r)
{
    const uint32_t c = static_cast<uint32_t>(q) + kSetSlack;
    return c < 64u * static_cast<uint32_t>(r) ? c : 64u * static_cast<uint32_t>(r);
}

// f(0) .. f(N - 1) with constant arguments.  (A loop over the registers with
// another loop inside is unrolled too late for its arrays to leave scratch
// memory: f16 rows at Q = 416 then took 13.3 ms in place of 10.1.)
template <class F, int... I>
__device__ __forceinline__ void static_for_(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for_(f, std::make_integer_sequence<int, N>{});
}

// R registers a lane.  kNan: keys may be NaN.
template <int R, bool kNan>
struct SetFrontier {
    static_assert(R >= 1 && R <= 8, "the heap operations hold 512 slots");
    static constexpr uint32_t kDone = UINT32_MAX;
    using Keys = uint32_t __attribute__((ext_vector_type(R)));
    Keys key;          // order key of a position; 0: free
    uint32_t unused;   // bit i: register i holds an unused entry
    uint2* entry;      // LDS [cap]: row, sample
    SplitHeap heap;    // LDS [Q + 2]: key and position
    uint64_t* log;     // this route's ring of admitted (position, key bits)
    uint32_t log_mask;
    uint32_t cap;
    int Q;
    // wave-uniform
    uint32_t logged, replayed;  // admissions so far; those the heap has seen
    int heap_size;              // slot 0 included
    int size;                   // entries of the frontier (those that have left excluded)
    uint32_t top;               // greatest key, its first position and the number of
    int top_pos, top_count;     // positions that hold it, once size == Q
    int top_gone;               // how many of those have left the frontier
    bool eager;

    __device__ void init(uint2* entry_, const SplitHeap& heap_, uint64_t* log_, uint32_t log_mask_,
                         int q)
    {
        static_for<R>([&](auto i) { key[int{i}] = 0u; });
        unused = 0u;
        entry = entry_;
        heap = heap_;
        log = log_;
        log_mask = log_mask_;
        cap = set_capacity(q, R);
        Q = q;
        logged = replayed = 0;
        heap_size = 1;
        size = 0;
        top = 0;
        top_pos = top_count = top_gone = 0;
        eager = false;
    }

    // Position pos takes key k (0: it is free).
    __device__ __forceinline__ void put(int pos, uint32_t k, bool is_unused, int lane)
    {
        const bool me = lane == (pos & (kWave - 1));
        static_for<R>([&](auto i) {
            if ((pos >> 6) == i) key[int{i}] = me ? k : key[int{i}];
        });
        const uint32_t bit = me ? 1u << (pos >> 6) : 0u;
        unused = is_unused ? unused | bit : unused & ~bit;
    }
    // The key of register i where its entry is unused.
    __device__ __forceinline__ uint32_t pick(int i, uint32_t k) const
    {
        return (unused >> i) & 1u ? k : kDone;
    }
    __device__ __forceinline__ int free_pos(int lane) const
    {
        int pos = -1;
        static_for<R>([&](auto r) {
            constexpr int i = R - 1 - r;
            const uint64_t m = ballot(key[int{i}] == 0u && static_cast<uint32_t>(64 * i + lane) < cap);
            if (m) pos = 64 * i + __builtin_ctzll(m);
        });
        return pos;
    }
    __device__ __forceinline__ void find_top()
    {
        uint32_t m = key[0];
        static_for<R>([&](auto i) { m = max(m, key[int{i}]); });
        top = wave_max_u32(m);
        top_count = 0;
        static_for<R>([&](auto r) {
            constexpr int i = R - 1 - r;
            const uint64_t at = ballot(key[int{i}] == top);
            top_count += __popcll(at);
            if (at) top_pos = 64 * i + __builtin_ctzll(at);
        });
    }

    // Brings the heap up to date with every admission so far, then takes the
    // positions of the greatest key's entries that have left, if any.  (The
    // log's stores are waited for: other lanes read them.)
    __device__ __forceinline__ void catch_up(int lane)
    {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        while (replayed < logged) {
            const uint32_t left = logged - replayed;
            const int n = left < static_cast<uint32_t>(kWave) ? static_cast<int>(left) : kWave;
            uint64_t e = 0;
            if (lane < n)
                e = __hip_atomic_load(log + ((replayed + static_cast<uint32_t>(lane)) & log_mask),
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const int lo = static_cast<int>(static_cast<uint32_t>(e));
            const int hi = static_cast<int>(static_cast<uint32_t>(e >> 32));
            for (int i = 0; i < n; ++i) {
                HeapPair p;
                p.first = __int_as_float(__builtin_amdgcn_readlane(lo, i));
                p.second = static_cast<uint32_t>(__builtin_amdgcn_readlane(hi, i));
                wave_smmh_insert(heap, heap_size, p, lane);
                if (heap_size >= Q + 2) (void)wave_smmh_pop_max(heap, heap_size, lane);
            }
            replayed += static_cast<uint32_t>(n);
        }
        __threadfence_block();
        if (top_gone == 0) return;
        static_for<R>([&](auto i) {
            for (uint64_t m = ballot(key[int{i}] == top); m; m &= m - 1) {
                const int l = __builtin_ctzll(m);
                bool in = false;
                for (int s = lane + 1; s < heap_size; s += kWave)
                    in |= heap.second[s] == static_cast<uint32_t>(64 * i + l);
                if (!ballot(in) && lane == l) {
                    key[int{i}] = 0u;
                    unused &= ~(1u << i);
                }
            }
        });
        top_gone = 0;
        find_top();
    }

    // The first entry (held by every lane), already marked used.
    __device__ __forceinline__ void seed(float first, uint32_t row, uint32_t sample, int lane)
    {
        const uint32_t k = order_key(first);
        if constexpr (kNan) {
            if (first != first) {
                eager = true;
                if (lane == 0) heap_set(heap, 1, HeapPair{first, 0u});
                heap_size = 2;
            }
        }
        place(0, 0, max(k, 1u), false, first, row, sample, lane);
        ++logged;
        size = 1;
    }

    // An admitted entry, held by lane j, takes position pos.
    __device__ __forceinline__ void place(int pos, int j, uint32_t k, bool is_unused, float first,
                                          uint32_t row, uint32_t sample, int lane)
    {
        if (lane == j) {
            entry[pos] = make_uint2(row, sample);
            if (!kNan || !eager)
                __hip_atomic_store(log + (logged & log_mask),
                                   (static_cast<uint64_t>(static_cast<uint32_t>(pos)) << 32) |
                                       __float_as_uint(first),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        put(pos, k, is_unused, lane);
    }

    // The ordered admission of one step: lane by lane, an entry enters unless
    // the frontier is full and its greatest key is less; past Q entries the
    // greatest leaves.  Returns the lanes admitted.
    __device__ __forceinline__ uint64_t admit(bool cand, float first, uint32_t row,
                                              uint32_t sample, int lane)
    {
        if constexpr (kNan) {
            if (!eager && ballot(cand && first != first)) {
                catch_up(lane);
                eager = true;
            }
            if (eager) return admit_eager(cand, first, row, sample, lane);
        }
        const uint32_t k = order_key(first);
        uint64_t adm = 0;
        for (uint64_t m = ballot(cand && !(size == Q && k > top)); m; m &= m - 1) {
            const int j = __builtin_ctzll(m);
            const uint32_t kj = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(k), j));
            if (size == Q && kj > top) continue;
            int pos;
            bool moved = true;  // the greatest key changes
            const bool over = size == Q && kj < top && top_count == 1;
            // the ring is full, or positions are all held by entries whose
            // leaving is open
            if (logged - replayed > log_mask || (size == Q && !over && free_pos(lane) < 0))
                catch_up(lane);
            if (over) {
                pos = top_pos;
            } else {
                if (size < Q) {
                    moved = ++size == Q;
                } else if (kj < top && top_gone + 1 == top_count) {
                    // the last entry of the greatest key leaves
                    static_for<R>([&](auto i) {
                        if (key[int{i}] == top) {
                            key[int{i}] = 0u;
                            unused &= ~(1u << i);
                        }
                    });
                    top_gone = 0;
                } else {
                    ++top_gone;
                    top_count += kj == top ? 1 : 0;
                    moved = false;
                }
                pos = free_pos(lane);
            }
            place(pos, j, kj, true, first, row, sample, lane);
            ++logged;
            adm |= 1ull << j;
            if (moved) find_top();
        }
        return adm;
    }

    // The same with every admission through the heap.
    __device__ __forceinline__ uint64_t admit_eager(bool cand, float first, uint32_t row,
                                                 uint32_t sample, int lane)
    {
        const uint32_t k = order_key(first);
        const bool full = heap_size >= Q + 1;
        const float thr = full ? heap.first[2] : 0.0f;
        float hmax = heap_size >= 3   ? heap.first[2]
                     : heap_size == 2 ? heap.first[1]
                                      : -__builtin_inff();
        uint64_t adm = 0;
        for (uint64_t m = ballot(cand && !(full && thr < first)); m; m &= m - 1) {
            const int j = __builtin_ctzll(m);
            HeapPair p;
            p.first = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(first), j));
            if (heap_size >= Q + 1 && hmax < p.first) continue;
            const uint32_t kj = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(k), j));
            const int pos = free_pos(lane);
            p.second = static_cast<uint32_t>(pos);
            place(pos, j, max(kj, 1u), true, first, row, sample, lane);
            wave_smmh_insert(heap, heap_size, p, lane);
            hmax = fmaxf(hmax, p.first);
            adm |= 1ull << j;
            if (heap_size >= Q + 2) {
                const int gone = __builtin_amdgcn_readfirstlane(static_cast<int>(heap.second[2]));
                hmax = wave_smmh_pop_max(heap, heap_size, lane);
                put(gone, 0u, false, lane);
            }
        }
        size = heap_size - 1;
        return adm;
    }

    // Of the unused entries of key mn, the position of lowest heap index.
    __device__ __forceinline__ int first_in_heap(uint32_t mn, int lane) const
    {
        for (int s0 = 1; s0 < heap_size; s0 += kWave) {
            const int s = s0 + lane;
            const uint32_t pos = s < heap_size ? heap.second[s] : 0u;
            uint32_t p = kDone;
            static_for<R>([&](auto i) {
                const uint32_t v = static_cast<uint32_t>(
                    __shfl(static_cast<int>(pick(i, key[int{i}])), static_cast<int>(pos & 63u), kWave));
                if ((pos >> 6) == static_cast<uint32_t>(i)) p = v;
            });
            const uint64_t m = ballot(s < heap_size && p == mn);
            if (m) return __builtin_amdgcn_readlane(static_cast<int>(pos), __builtin_ctzll(m));
        }
        return 0;  // not reached: an unused entry is in the heap
    }

    // The next entry (marked used); false when every entry is used.
    __device__ __forceinline__ bool pickup(Entry& out, int lane)
    {
        for (;;) {
            uint32_t p = kDone;
            static_for<R>([&](auto i) { p = min(p, pick(i, key[int{i}])); });
            const uint32_t mn = wave_min_u32(p);
            int ties = 0, pos = 0;
            static_for<R>([&](auto r) {
                constexpr int i = R - 1 - r;
                const uint64_t at = ballot(pick(i, key[int{i}]) == mn);
                ties += __popcll(at);
                if (at) pos = 64 * i + __builtin_ctzll(at);
            });
            if (mn == kDone) return false;
            const bool open = top_gone > 0 && mn == top;
            if (open || ties > 1) {
                if (!kNan || !eager) catch_up(lane);
                if (open) continue;
                pos = first_in_heap(mn, lane);
            }
            const uint2 rs = entry[pos];
            out.first = order_key_float(mn);
            out.second = rs.x;
            out.sample = rs.y;
            out.base = out.first;
            if (lane == (pos & (kWave - 1))) unused &= ~(1u << (pos >> 6));
            return true;
        }
    }
};

// Entries of a route's log ring: admissions between two looks at the heap
// (a full ring brings the heap up to date).  Whole routes admitted 350 at
// Q = 72 and 1260 at Q = 416.
inline uint32_t set_log_entries(int q) { return q <= 112 ? 1024u : 2048u; }

// The context keeps its rings from call to call; a launch of more routes
// (131,072 at Q > 112) takes the heap frontier.
constexpr size_t kSetLogBytes = size_t{2} << 30;

// Registers a lane for a beam of q, with the log rings of `routes` launch
// slots, or 0 where the heap frontier runs instead: beams that the wave heap
// operations do not hold, or no buffer for the rings (optional_scratch).
inline int set_registers(Context* ctx, int q, uint32_t routes, uint64_t** log)
{
    const int regs = q + static_cast<int>(kSetSlack) <= 128   ? 2
                     : q + static_cast<int>(kSetSlack) <= 256 ? 4
                     : q + static_cast<int>(kSetSlack) <= 512 ? 8
                                                              : 0;
    if (regs == 0) return 0;
    const size_t bytes = static_cast<size_t>(routes) * set_log_entries(q) * sizeof(uint64_t);
    if (bytes > kSetLogBytes) return 0;
    *log = static_cast<uint64_t*>(ctx->optional_scratch(Context::kScratchLog, bytes));
    return *log != nullptr ? regs : 0;
}

}  // namespace gofann
