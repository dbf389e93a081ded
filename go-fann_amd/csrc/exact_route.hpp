// exact_route.hpp -- device side of the full-GPU exact-distance route: the
// route of exact_route.hip, its arguments and its launch, shared by the
// kernels with the heap frontier (exact_route.hip) and those with the set
// frontier (exact_set_*.hip, one source per element type).
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>
#include <string>

#include "device_common.hpp"
#include "exact_dist.hpp"
#include "gofann_internal.hpp"
#include "set_frontier.hpp"

namespace gofann {

constexpr int kExactMaxTopk = 10;  // defaults::max_topk

// 1: rows of 128, 192 or 256 bytes use kernels with the row length fixed
// at compile time (all of a row's loads in flight at once, at the price of
// about 40 more VGPRs and so fewer resident routes); 0 keeps the loop.
#ifndef GOFANN_EXACT_FIXED_ROWS
#define GOFANN_EXACT_FIXED_ROWS 0
#endif

// Minimum waves per SIMD the u8 kernels are compiled for (register budget).
// 6 holds them to 80 VGPRs, 24 routes per CU, without spills (the lane id and
// the arguments are taken anew per step).  At C2, Q = 80: 46.1 ms, against 49.0
// at 5 waves and 54.1 at 7 (the visited table leaves LDS).  The f32 / f16 kernels
// (eight partial sums and two 16-byte loads per lane) take fewer (below).
#ifndef GOFANN_EXACT_MIN_WAVES
#define GOFANN_EXACT_MIN_WAVES 6
#endif

// 16-byte row chunks loaded per memory round trip in the any-dim row loop.
// With one chunk's query words in registers at a time four fit the 80 VGPRs
// without spills; 57,000 routes of 192 bytes, Q = 72: three take 13.6 ms, four
// 12.5, six (four registers spilled) 12.5.
#ifndef GOFANN_EXACT_ROW_UNROLL
#define GOFANN_EXACT_ROW_UNROLL 4
#endif

// Waves per SIMD the f32 / f16 kernels are compiled for, and the 128-byte
// blocks per quad whose loads are issued before any is summed.  The quad
// kernels are bound by the loads in flight; their LDS holds them near 4
// waves per SIMD anyway (C4, 1 KB f16 rows, Q = 448: 17 routes per CU), so
// they take the registers for deeper batches: exact route 141.6 ms with two
// blocks left to the compiler's unrolling at 5 waves, 119.0 with explicit
// batches of two, 110.1 with batches of four at 4 waves (no spills; eight
// spill 8-14 VGPRs).
#ifndef GOFANN_EXACT_FLOAT_MIN_WAVES
#define GOFANN_EXACT_FLOAT_MIN_WAVES 4
#endif
#ifndef GOFANN_EXACT_QUAD_UNROLL
#define GOFANN_EXACT_QUAD_UNROLL 4
#endif
constexpr int kExactQuadUnroll = GOFANN_EXACT_QUAD_UNROLL;

struct ExactArgs {
    gofann_graph_view graph;
    const uint32_t* label_size;
    gofann_predicate_view pred;
    gofann_routes routes;
    const uint8_t* base;
    const uint8_t* queries;
    uint32_t dim;
    uint32_t samples;
    gofann_exact_params params;
    uint32_t* out_ids;
    float* out_dists;
    gofann_route_stats* stats;
    uint32_t* hash_global;
    uint32_t off_frontier;
    uint32_t off_hash;
    uint32_t off_heap;   // set frontier: its heap, and the routes' log rings
    uint64_t* log;
    uint32_t log_mask;
};

// Squared L2 of a u8 row against the query held in LDS (q, |q|^2); kU
// 16-byte chunks per memory round trip when dim is a multiple of 16.
template <int kU>
__device__ __forceinline__ uint32_t l2_u8_row(const uint8_t* row, const uint32_t* q,
                                              uint32_t dim, uint32_t qnorm)
{
    uint32_t nb = 0, dot = 0;
    if ((dim & 15u) == 0) {
        const uint4* r4 = reinterpret_cast<const uint4*>(row);
        const uint4* q4 = reinterpret_cast<const uint4*>(q);
        const auto add = [&](const uint4& b, uint32_t i) {
            const uint4 w = q4[i];
            nb = __builtin_amdgcn_udot4(b.x, b.x, nb, false);
            nb = __builtin_amdgcn_udot4(b.y, b.y, nb, false);
            nb = __builtin_amdgcn_udot4(b.z, b.z, nb, false);
            nb = __builtin_amdgcn_udot4(b.w, b.w, nb, false);
            dot = __builtin_amdgcn_udot4(b.x, w.x, dot, false);
            dot = __builtin_amdgcn_udot4(b.y, w.y, dot, false);
            dot = __builtin_amdgcn_udot4(b.z, w.z, dot, false);
            dot = __builtin_amdgcn_udot4(b.w, w.w, dot, false);
        };
        const uint32_t n = dim / 16;
        uint32_t i = 0;
        for (; i + kU <= n; i += kU) {
            uint4 b[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) b[u] = r4[i + u];
            // one chunk's query words in registers at a time
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                add(b[u], i + u);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        for (; i < n; ++i) add(r4[i], i);
        return nb + qnorm - 2u * dot;
    }
    if ((dim & 3u) == 0) {
        const uint32_t* r1 = reinterpret_cast<const uint32_t*>(row);
        for (uint32_t i = 0; i < dim / 4; ++i) {
            const uint32_t b = r1[i];
            nb = __builtin_amdgcn_udot4(b, b, nb, false);
            dot = __builtin_amdgcn_udot4(b, q[i], dot, false);
        }
        return nb + qnorm - 2u * dot;
    }
    const uint8_t* qb = reinterpret_cast<const uint8_t*>(q);
    uint32_t acc = 0;
    for (uint32_t d = 0; d < dim; ++d) {
        const int diff = static_cast<int>(row[d]) - static_cast<int>(qb[d]);
        acc += static_cast<uint32_t>(diff * diff);
    }
    return acc;
}

// Rows of kC 16-byte chunks (dim = 16 kC): every chunk's load is issued
// before the first dot product, so a row costs one memory round trip.
template <int kC>
__device__ __forceinline__ void row_load(const uint8_t* row, bool keep, uint4 (&b)[kC])
{
    const uint4* r4 = reinterpret_cast<const uint4*>(row);
#pragma unroll
    for (int i = 0; i < kC; ++i) b[i] = keep ? r4[i] : make_uint4(0, 0, 0, 0);
}

template <int kC>
__device__ __forceinline__ uint32_t row_dist(const uint4 (&b)[kC], const uint32_t* q,
                                             uint32_t qnorm)
{
    const uint4* q4 = reinterpret_cast<const uint4*>(q);
    uint32_t nb = 0, dot = 0;
#pragma unroll
    for (int i = 0; i < kC; ++i) {
        const uint4 w = q4[i];
        nb = __builtin_amdgcn_udot4(b[i].x, b[i].x, nb, false);
        nb = __builtin_amdgcn_udot4(b[i].y, b[i].y, nb, false);
        nb = __builtin_amdgcn_udot4(b[i].z, b[i].z, nb, false);
        nb = __builtin_amdgcn_udot4(b[i].w, b[i].w, nb, false);
        dot = __builtin_amdgcn_udot4(b[i].x, w.x, dot, false);
        dot = __builtin_amdgcn_udot4(b[i].y, w.y, dot, false);
        dot = __builtin_amdgcn_udot4(b[i].z, w.z, dot, false);
        dot = __builtin_amdgcn_udot4(b[i].w, w.w, dot, false);
    }
    return nb + qnorm - 2u * dot;
}

__device__ __forceinline__ bool better(float ld, uint32_t lid, float rd, uint32_t rid)
{
    return ld < rd || (ld == rd && lid < rid);
}

// insert_best_result (backend_full_gpu.cu:1342-1375) on a register array:
// lane i < K holds entry i, ascending by (distance, id), ids unique.  Every
// lane calls it with the same (d, id); size is wave-uniform.  The entries
// live in the first 16-lane row (K <= 10), so shifts are row DPP moves.
struct BestK {
    float d;
    uint32_t id;
};

__device__ __forceinline__ uint32_t dpp_u32(uint32_t v, int ctrl)
{
    switch (ctrl) {
    case 0x101: return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x101, 0xF, 0xF, false));
    default: return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x111, 0xF, 0xF, false));
    }
}

__device__ __forceinline__ bool best_insert(BestK& b, float d, uint32_t id, uint32_t K,
                                            uint32_t& size, int lane)
{
    const bool in = static_cast<uint32_t>(lane) < size;
    const uint64_t dup = ballot(in && b.id == id);
    if (dup) {
        const int i = __builtin_ctzll(dup);
        if (d >= __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b.d), i))) return false;
        // drop entry i: lanes i.. take their right neighbour (row_shl:1)
        const uint32_t nd = dpp_u32(__float_as_uint(b.d), 0x101);
        const uint32_t ni = dpp_u32(b.id, 0x101);
        if (lane >= i) {
            b.d = __uint_as_float(nd);
            b.id = ni;
        }
        --size;
    }
    if (size == K) {
        const float ld = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b.d), static_cast<int>(K) - 1));
        const uint32_t li = static_cast<uint32_t>(
            __builtin_amdgcn_readlane(static_cast<int>(b.id), static_cast<int>(K) - 1));
        if (!better(d, id, ld, li)) return false;
    }
    // entries before (d, id) stay; the rest move right (row_shr:1)
    const int pos = __popcll(ballot(static_cast<uint32_t>(lane) < size && better(b.d, b.id, d, id)));
    const uint32_t sd = dpp_u32(__float_as_uint(b.d), 0x111);
    const uint32_t si = dpp_u32(b.id, 0x111);
    if (lane > pos) {
        b.d = __uint_as_float(sd);
        b.id = si;
    } else if (lane == pos) {
        b.d = d;
        b.id = id;
    }
    if (size < K) ++size;
    return true;
}

// Loads a picked node needs when it is expanded, issued at pickup: lane j's
// adjacency entry j (and its sample id when the graph carries them), and the
// node's label slab or CSR bounds (.x/.y) for the filter.
struct ExactNode {
    uint32_t adj;
    uint32_t nsamp;
    uint4 row;
};

__device__ __forceinline__ void load_node(const gofann_graph_view& g,
                                          const gofann_predicate_view& pv, bool verdict_rows,
                                          uint32_t off, uint32_t degree, const Entry& e, int lane,
                                          ExactNode& n)
{
    const size_t row = static_cast<size_t>(off + (e.second & ~kPoolUsed)) * g.degree;
    const bool in_row = static_cast<uint32_t>(lane) < degree;
    n.adj = in_row ? g.graph[row + lane] : UINT32_MAX;
    n.nsamp = (in_row && g.neighbor_samples) ? g.neighbor_samples[row + lane] : 0u;
    n.row = make_uint4(0, 0, 0, 0);
    if (verdict_rows && e.sample < pv.rows && pv.csr_offsets != nullptr) {
        if (slab_usable(pv, e.sample)) {
            n.row = slab_load(pv, e.sample);
        } else {
            n.row.x = pv.csr_offsets[e.sample];
            n.row.y = pv.csr_offsets[e.sample + 1];
        }
    }
}

// Float rows (f32 / f16): the neighbours' exact distances in the warp
// order; lane j of the wave returns the distance of its own candidate
// (FLT_MAX where keep is false).  Rows up to kQuadMaxRowBytes: 16 rows at a
// time, one per quad of lanes (l2_w32_quad), candidates compacted through
// LDS in lane order (s_samp and s_dist, kMaxDegree entries, are free at
// this point of the step).  Longer rows (kLong, its own kernel): two at a
// time, one per 32-lane half (l2_w32_partial + w32_tree), which keeps every
// lane busy, with kExactLongBatch row words per lane in flight: at C3's
// 16 KB rows 181 ms a step for the graph routes, against 269 with 8 words
// and 348 for the quads; at C4's 1 KB rows the quads (then two blocks a
// lane in flight) took 140 against 329 for the halves.  Either form gives
// the same bits for any row length.
constexpr size_t kQuadMaxRowBytes = 4096;

#ifndef GOFANN_EXACT_LONG_BATCH
#define GOFANN_EXACT_LONG_BATCH 32
#endif
constexpr int kExactLongBatch = GOFANN_EXACT_LONG_BATCH;

template <int kElem, bool kLong>
__device__ __forceinline__ float wave_float_dists(const uint8_t* base, uint32_t dim,
                                                  const float* qf, bool keep, uint32_t samp,
                                                  int lane, uint32_t* s_samp, float* s_dist)
{
    const size_t row_bytes = static_cast<size_t>(dim) * elem_bytes(kElem);
    uint64_t m = ballot(keep);
    if constexpr (kLong) {
        float out = FLT_MAX;
        while (m) {
            const int ja = __builtin_ctzll(m);
            m &= m - 1;
            int jb = -1;
            if (m) {
                jb = __builtin_ctzll(m);
                m &= m - 1;
            }
            const uint32_t sa = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(samp), ja));
            const uint32_t sb =
                jb >= 0 ? static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(samp), jb))
                        : sa;
            const uint32_t s = lane < 32 ? sa : sb;
            const float t = w32_tree<kElem>(l2_w32_partial<kElem, kExactLongBatch>(
                base + static_cast<size_t>(s) * row_bytes, qf, dim, static_cast<uint32_t>(lane) & 31u));
            const float da = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t), 0));
            const float db = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t), 32));
            if (lane == ja) out = da;
            if (lane == jb) out = db;
        }
        return out;
    }
    const int n = __popcll(m);
    const uint32_t rank = lanes_below(m);
    if (keep) s_samp[rank] = samp;
    __threadfence_block();
    const int quad = lane >> 2;
    const uint32_t g = static_cast<uint32_t>(lane) & 3u;
    for (int c = quad; c - quad < n; c += 16) {
        if (c < n) {
            const uint32_t s = s_samp[c];
            const float d = l2_w32_quad<kElem, kExactQuadUnroll>(
                base + static_cast<size_t>(s) * row_bytes, qf, dim, g);
            if (g == 0) s_dist[c] = d;
        }
    }
    __threadfence_block();
    return keep ? s_dist[rank] : FLT_MAX;
}

// kC > 0 (u8): dim == 16 kC (rows loaded whole); kC == 0: any dim; kC < 0
// (f32 / f16): rows longer than kQuadMaxRowBytes.  The frontier lives in
// LDS.  kElem: the element type of base and queries
// (GOFANN_ELEM_*); u8 rows are scored per lane (integer, exact in any
// order), f32 / f16 rows by wave_float_dists.
// kR: 0, the frontier is the heap in LDS; else a set of kR registers a lane
// (set_frontier.hpp).
template <int kVisited, int kC, int kElem, int kR>
__device__ __forceinline__ void exact_route(const ExactArgs& args, unsigned char* lds)
{
    constexpr int kRowUnroll = GOFANN_EXACT_ROW_UNROLL;
    constexpr bool kSet = kR > 0;
    __shared__ uint32_t s_row[kMaxDegree];
    __shared__ uint32_t s_samp[kMaxDegree];
    __shared__ float s_dist[kMaxDegree];
    __shared__ uint64_t s_adm;

    const ExactArgs& a = args;
    const int lane = static_cast<int>(threadIdx.x);
    const uint32_t slot = xcd_slot(blockIdx.x, gridDim.x);
    if (slot >= a.routes.count) return;
    const uint32_t route = a.routes.launch_order ? a.routes.launch_order[slot] : slot;
    const int Q = a.params.queue_limit;
    const uint32_t K = static_cast<uint32_t>(a.params.topk);
    const int mode = a.params.early_stop_mode;

    uint32_t* qw = reinterpret_cast<uint32_t*>(lds);
    Entry* frontier = reinterpret_cast<Entry*>(lds + a.off_frontier);
    SetFrontier<kSet ? kR : 1, kElem != GOFANN_ELEM_U8> set;
    VisitedSet<kVisited> visited;

    const uint32_t group = a.routes.route_group[route];
    const uint32_t seed = a.routes.route_start[route];
    const uint32_t gsize = a.label_size ? a.label_size[group] : UINT32_MAX;
    const uint32_t off = a.graph.label_offset[group];
    const uint64_t qfbit = a.routes.query_filter_bits ? a.routes.query_filter_bits[route] : ~0ULL;
    const uint32_t active = count_active_ranges(a.routes.range_modes, route, a.routes.range_count);
    const bool enabled = pred_enabled(a.pred, route);
    const uint32_t degree = a.graph.degree < static_cast<uint32_t>(kMaxDegree)
                                ? a.graph.degree
                                : static_cast<uint32_t>(kMaxDegree);

    // Query row into LDS: u8 as words (zero-padded to 16 bytes) with |q|^2,
    // f32 / f16 as f32.
    const float* qf = reinterpret_cast<const float*>(lds);
    uint32_t qn = 0;
    if constexpr (kElem == GOFANN_ELEM_U8) {
        const uint8_t* qrow = a.queries + static_cast<size_t>(a.routes.route_query[route]) * a.dim;
        const uint32_t qwords = (a.dim + 15u) / 16u * 4u;
        for (uint32_t w = lane; w < qwords; w += kWave) {
            uint32_t v = 0;
            for (uint32_t b = 0; b < 4; ++b) {
                const uint32_t d = w * 4 + b;
                if (d < a.dim) v |= static_cast<uint32_t>(qrow[d]) << (8 * b);
            }
            qw[w] = v;
            qn = __builtin_amdgcn_udot4(v, v, qn, false);
        }
        for (int o = 32; o > 0; o >>= 1) qn += static_cast<uint32_t>(__shfl_xor(static_cast<int>(qn), o, kWave));
    } else {
        const uint8_t* qrow = a.queries + static_cast<size_t>(a.routes.route_query[route]) * a.dim *
                                              elem_bytes(kElem);
        float* qs = reinterpret_cast<float*>(lds);
        for (uint32_t d = lane; d < a.dim; d += kWave) qs[d] = elem_to_float<kElem>(qrow, d);
    }
    visited.init(reinterpret_cast<uint32_t*>(lds + a.off_hash),
                 a.hash_global ? a.hash_global + static_cast<size_t>(slot) * kHashCapacity : nullptr,
                 lane);
    __threadfence_block();
    __syncthreads();

    gofann_route_stats st{0, 0, 0, 0, 0, 0, 0, 0};
    PredCounters pc{0, 0};
    uint32_t bsize = 0;  // wave-uniform
    BestK bk{FLT_MAX, UINT32_MAX};
    int heap_size = 1;
    bool done = false;
    const Entry sentinel = {FLT_MAX, UINT32_MAX, FLT_MAX, UINT32_MAX};
    Entry now = sentinel, next = sentinel;

    // Seed (:1793-1850).
    if (gsize == 0 || seed == UINT32_MAX || seed >= gsize) {
        done = true;
    } else {
        const uint32_t s0 = a.graph.row_to_sample[off + seed];
        if (s0 < a.samples) {
            float d0;
            if constexpr (kElem == GOFANN_ELEM_U8) {
                d0 = bcast0f(lane == 0 ? static_cast<float>(l2_u8_row<kRowUnroll>(
                                             a.base + static_cast<size_t>(s0) * a.dim, qw, a.dim, qn))
                                       : 0.0f);
            } else {
                // every quad scores the seed row; lane 0's sum is it
                d0 = bcast0f(l2_w32_quad<kElem>(
                    a.base + static_cast<size_t>(s0) * a.dim * elem_bytes(kElem), qf, a.dim,
                    static_cast<uint32_t>(lane) & 3u));
            }
            const Entry kp = {d0, seed, d0, s0};
            if constexpr (kSet) {
                set.init(reinterpret_cast<uint2*>(lds + a.off_frontier),
                         split_heap(lds + a.off_heap, Q),
                         a.log + static_cast<size_t>(slot) * (a.log_mask + 1), a.log_mask, Q);
                set.seed(d0, seed, s0, lane);
                now = kp;
            } else {
                if (lane == 0) smmh_insert(frontier, heap_size, kp);
                heap_size = bcast0(heap_size);
            }
            if (lane == 0) (void)visited.add_serial(seed, 0);
            visited.count = 1;
            st.scored = 1;
        } else {
            done = true;
        }
    }
    __threadfence_block();
    __syncthreads();
    if constexpr (!kSet) {  // (the set's seed is the first entry picked)
        if (!done && !pickup(frontier, heap_size, now, lane)) done = true;
    }
    if (done) st.exhausted = 1;

    ExactNode cur{UINT32_MAX, 0, make_uint4(0, 0, 0, 0)};
    if (!done) load_node(a.graph, a.pred, enabled, off, degree, now, lane, cur);

    uint32_t steps = 0, finished = 0;
    bool first_step = true;
    const int wave_lane = lane;
    while (!done) {
        // per step: lane-derived values are not held across steps (no spills
        // at 6 waves; with the lane hoisted out of the loop, 10 VGPRs spilled),
        const int lane = opaque_lane(wave_lane);
        // nor are the arguments (held over the route, 105-128 scalar registers
        // were spilled into vector lanes; read per step, 6-21 in the heap's
        // kernels and 19-53 in the set's)
        const ExactArgs& a = step_args<ExactArgs>();
        if (a.params.max_steps != 0 && steps >= static_cast<uint32_t>(a.params.max_steps)) break;

        // One memory round for the neighbours (visited tests, sample ids) and
        // the expanded node's label row, then one for the neighbours' rows.
        const uint32_t adj = cur.adj;
        const bool fresh = adj != UINT32_MAX && adj < gsize && !visited.test(adj);
        uint32_t samp = 0;
        if (fresh) samp = a.graph.neighbor_samples ? cur.nsamp : a.graph.row_to_sample[off + adj];
        const bool keep = fresh && samp < a.samples;
        const uint32_t sample = now.sample;
        WaveRow vrow{0, 0, UINT32_MAX, false};
        if (enabled) {
            if (!slab_usable(a.pred, sample)) {
                vrow = wave_row_load(a.pred, sample, cur.row.x, cur.row.y, lane);
            } else if (slab_count(cur.row) != kSlabOverflow) {
                vrow = wave_row_from_slab(cur.row, lane);
            } else {
                vrow = wave_row_load(a.pred, sample, a.pred.csr_offsets[sample],
                                     a.pred.csr_offsets[sample + 1], lane);
            }
        }
        uint32_t d32 = 0;
        float fdist = FLT_MAX;
        if constexpr (kElem == GOFANN_ELEM_U8) {
            const uint8_t* brow = a.base + static_cast<size_t>(samp) * a.dim;
            if constexpr (kC > 0) {
                uint4 rb[kC];
                row_load<kC>(brow, keep, rb);
                d32 = row_dist<kC>(rb, qw, qn);
            } else {
                d32 = keep ? l2_u8_row<kRowUnroll>(brow, qw, a.dim, qn) : 0u;
            }
            // The distance is complete here: the rows and query words are
            // dead before the filter below.
            asm volatile("" : "+v"(d32)::"memory");
        } else {
            fdist = wave_float_dists<kElem, (kC < 0)>(a.base, a.dim, qf, keep, samp, lane, s_samp,
                                                       s_dist);
            asm volatile("" : "+v"(fdist)::"memory");
        }

        // The expanded node's filter (wave-uniform) and best-k (lane 0).
        const uint32_t grow = off + (now.second & ~kPoolUsed);
        const uint64_t rmask = a.routes.row_filter_mask ? a.routes.row_filter_mask[grow] : ~0ULL;
        bool ok = (rmask & qfbit) != 0;
        if (ok && active != 0) ok = count_matching_ranges(a.routes, route, sample) == active;
        PredCounters c{0, 0};
        if (ok && enabled) ok = wave_pred_matches(a.pred, route, sample, vrow, lane, c);
        int improved = 0;
        if (lane == 0) {
            pc.rows += c.rows;
            pc.labels += c.labels;
        }
        if (ok) improved = best_insert(bk, now.first, sample, K, bsize, lane) ? 1 : 0;
        ++st.expanded;
        st.passed += ok ? 1 : 0;
        ++steps;

        const float dist = kElem == GOFANN_ELEM_U8 ? (keep ? static_cast<float>(d32) : FLT_MAX)
                                                   : fdist;
        st.scored += __popcll(ballot(keep));

        // Drop what cannot enter a full frontier (its maximum only falls
        // during the step), then admit the rest in adjacency order.
        uint64_t adm = 0;  // admitted lanes
        if constexpr (kSet) {
            adm = set.admit(keep, dist, adj, samp, lane);
        } else {
            const bool full = heap_size > 2 && heap_size >= Q + 1;
            const float thr = full ? frontier[2].first : 0.0f;
            const bool cand = keep && !(full && thr < dist);
            const uint64_t cand_mask = ballot(cand);
            if (Q + 2 <= kWaveHeapSlots) {
                // the whole wave runs each heap operation (same array as the
                // lane-0 sifts below); hmax: the largest `first` in the heap
                float hmax = heap_size >= 3   ? frontier[2].first
                             : heap_size == 2 ? frontier[1].first
                                              : -__builtin_inff();
                for (uint64_t m = cand_mask; m; m &= m - 1) {
                    const int j = __builtin_ctzll(m);
                    Entry kp;
                    kp.first = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dist), j));
                    kp.second = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(adj), j));
                    kp.sample = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(samp), j));
                    kp.base = kp.first;
                    if (heap_size > 2 && heap_size >= Q + 1 && hmax < kp.first) continue;
                    wave_smmh_insert(frontier, heap_size, kp, lane);
                    hmax = fmaxf(hmax, kp.first);
                    adm |= 1ull << j;
                    if (heap_size >= Q + 2) hmax = wave_smmh_pop_max(frontier, heap_size, lane);
                }
            } else {
                const int n_cand = __popcll(cand_mask);
                const uint32_t pos = lanes_below(cand_mask);
                if (cand) {
                    s_row[pos] = adj;
                    s_samp[pos] = samp;
                    s_dist[pos] = dist;
                }
                __syncthreads();
                if (lane == 0) {
                    uint64_t ap = 0;
                    for (int i = 0; i < n_cand; ++i) {
                        const Entry kp = {s_dist[i], s_row[i], s_dist[i], s_samp[i]};
                        if (heap_size > 2 && heap_size >= Q + 1 && frontier[2].first < kp.first)
                            continue;
                        smmh_insert(frontier, heap_size, kp);
                        ap |= 1ull << i;
                        if (heap_size >= Q + 2) smmh_pop_max(frontier, heap_size);
                    }
                    s_adm = ap;
                }
                heap_size = bcast0(heap_size);
                __syncthreads();
                const uint64_t ap = s_adm;  // by compacted position
                adm = ballot(cand && ((ap >> pos) & 1ull));
            }
        }
        const uint32_t n_adm = static_cast<uint32_t>(__popcll(adm));
        st.admitted += static_cast<int32_t>(n_adm);
        visited.reserve(n_adm, lane);
        if (visited.count + n_adm <= kHashCapacity) {
            const int ins = ((adm >> lane) & 1ull) ? visited.add_parallel(adj) : 0;
            visited.count += static_cast<uint32_t>(__popcll(ballot(ins != 0)));
        } else {
            // The set may fill: serial adds in admission (lane) order
            // reproduce which values the reference drops.
            uint32_t added = 0;
            for (uint64_t m = adm; m; m &= m - 1) {
                const int j = __builtin_ctzll(m);
                const uint32_t v = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(adj), j));
                if (lane == 0) added += static_cast<uint32_t>(visited.add_serial(v, added));
            }
            visited.count += bcast0u(added);
        }
        __threadfence_block();
        __syncthreads();

        // Pickup and early stop (:1985-2030).
        bool found;
        if constexpr (kSet) {
            found = set.pickup(next, lane);
        } else {
            found = pickup(frontier, heap_size, next, lane);
        }
        if (!found) {
            st.exhausted = 1;
            break;
        }
        load_node(a.graph, a.pred, enabled, off, degree, next, lane, cur);
        int stop = 0;
        const float kd = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(bk.d), static_cast<int>(K) - 1));
        const uint32_t ki = static_cast<uint32_t>(
            __builtin_amdgcn_readlane(static_cast<int>(bk.id), static_cast<int>(K) - 1));
        if (lane == 0 && !first_step) {
            if (mode == GOFANN_EARLY_STOP_ADAPTIVE && improved) {
                finished = 0;
            } else if (bsize == K && !better(next.first, next.sample, kd, ki)) {
                ++finished;
                stop = early_stop_reached(mode, static_cast<int>(finished), a.params.finish_limit,
                                          Q, st.expanded, st.passed, static_cast<int>(K))
                           ? 1
                           : 0;
            } else {
                finished = 0;
            }
        }
        if (bcast0(stop)) break;
        now = next;
        first_step = false;
    }

    __syncthreads();
    uint32_t* oid = a.out_ids + static_cast<size_t>(route) * K;
    float* od = a.out_dists + static_cast<size_t>(route) * K;
    const uint32_t nb = bsize;
    if (static_cast<uint32_t>(lane) < K) {
        oid[lane] = static_cast<uint32_t>(lane) < nb ? bk.id : UINT32_MAX;
        od[lane] = static_cast<uint32_t>(lane) < nb ? bk.d : FLT_MAX;
    }
    const int pred_rows = wave_sum(static_cast<int>(pc.rows));
    const int pred_labels = wave_sum(static_cast<int>(pc.labels));
    if (lane == 0 && a.stats) {
        st.steps = static_cast<int32_t>(steps);
        st.pred_rows = pred_rows;
        st.pred_labels = pred_labels;
        a.stats[route] = st;
    }
}

// The kernels: one wave64 per route.
template <int kVisited, int kC, int kElem>
__global__ __launch_bounds__(64, (kElem == GOFANN_ELEM_U8 ? GOFANN_EXACT_MIN_WAVES : GOFANN_EXACT_FLOAT_MIN_WAVES)) void exact_route_kernel(ExactArgs a)
{
    extern __shared__ __align__(16) unsigned char lds[];
    exact_route<kVisited, kC, kElem, 0>(a, lds);
}

// Waves per SIMD a set kernel is compiled for.  With four, two of its kinds
// ran out of registers: f16 with the full LDS table spilled 16 at R = 2 (with
// two waves' registers it takes 133, and the table leaves at most nine routes a
// CU anyway; dim 512, Q = 64, 280 routes: 1.28 -> 1.22 ms), and long f32 rows at
// R = 8 were scheduled into 95, the query read from LDS word by word between
// the sums (with three waves' registers the reads go out ahead in 126, still
// four waves; 2.7M rows of 16 KB, 6,666 routes at Q = 256 and 352: 187 -> 168 ms).
template <int kVisited, int kC, int kElem>
constexpr int set_min_waves()
{
    if (kElem == GOFANN_ELEM_F16 && kVisited == kVisitedLds) return 2;
    return kElem == GOFANN_ELEM_F32 && kC < 0 ? 3 : 4;
}

template <int kVisited, int kC, int kElem, int kR>
__global__ __launch_bounds__(64, (set_min_waves<kVisited, kC, kElem>())) void exact_set_kernel(ExactArgs a)
{
    extern __shared__ __align__(16) unsigned char lds[];
    exact_route<kVisited, kC, kElem, kR>(a, lds);
}

template <int kVisited, int kC, int kElem, int kR>
constexpr auto exact_kernel()
{
    if constexpr (kR == 0)
        return &exact_route_kernel<kVisited, kC, kElem>;
    else
        return &exact_set_kernel<kVisited, kC, kElem, kR>;
}

template <int kVisited, int kC, int kElem, int kR>
int exact_resident(Context* ctx, uint32_t lds)
{
    return resident_blocks(
        ctx, reinterpret_cast<const void*>(exact_kernel<kVisited, kC, kElem, kR>()), lds);
}

// Whether the spilling table pays where the slab holds up to a third more
// routes.  u8 rows: narrow beams (at Q <= 72 also launches of more than one
// round of resident routes), and launches of more than two rounds where the
// rows' own traffic is high (degree x dim of 8 KB a step or more), which the
// slabs' (16 KB a route) adds to.  The spilling table (24 routes a CU up to Q =
// 80, 21 to Q = 128) against the slab (28), ms at dim x degree:
//   89 x 64, 2,800 routes, 1,800 rows a group: Q = 64 0.71 / 0.86, Q = 111 1.12 /
//     1.31, Q = 160 1.60 / 1.78, Q = 224 2.50 / 2.40; 7,400 rows: Q = 160 1.87 / 1.95,
//     Q = 224 3.36 / 2.62; 14,800: Q = 111 1.61 / 1.64, Q = 160 2.36 / 2.20; 44,000:
//     Q = 64 1.36 / 1.41, Q = 111 2.44 / 1.99
//   192 x 64, Q = 32: 3,000 routes 0.89 / 0.92, 12,000 1.52 / 1.76
//   192 x 64, Q = 72: 5,000 routes 2.07 / 1.99, 20,000 5.02 / 5.68, 57,000
//     11.7 / 14.2; Q = 96: 2.53 / 2.43, 6.77 / 7.13, 16.5 / 17.8; 12,000 at
//     Q = 112 4.36 / 4.07; 57,000 at Q = 128 21.8 / 22.2
//   96 x 32, Q = 64: 6,000 1.84 / 1.81, 45,000 8.13 / 8.34; Q = 96: 2.94 /
//     2.38, 12.5 / 11.5
//   96 x 64, Q = 96: 12,000 4.43 / 3.84, 45,000 12.1 / 12.1; 128 x 48: 45,000
//     12.0 / 11.0
// Float rows: narrow beams of launches that the spilling table holds (f32 dim
// 640, Q = 224, 14 against 16 a CU: 1,800 rows a group 4.48 / 4.87, 14,800 rows 5.90 /
// 5.48); f16 dim 512, Q = 416, 12 against 16: 12.4 / 10.9; f32 rows of 16 KB, Q = 352,
// 6 against 7: 186 / 181.
template <int kElem>
bool spill_pays(const Context* ctx, const ExactArgs& a, uint32_t count, int spilling,
                int residents)
{
    if (kElem != GOFANN_ELEM_U8)
        return a.params.queue_limit <= narrow_beam(a.graph, 224, 160, 160) &&
               all_resident(ctx, count, spilling);
    if (a.params.queue_limit <= narrow_beam(a.graph, 160, 112, 64)) return true;
    const uint64_t round = static_cast<uint64_t>(residents) * static_cast<uint64_t>(ctx->compute_units);
    if (a.params.queue_limit <= 72) return count > round;
    return count > 2 * round && static_cast<uint64_t>(a.dim) * a.graph.degree >= 8192;
}

// Visited-set placement, then the launch.  Auto: the full LDS table where
// full_table says so, else the most resident routes per CU, LDS preferred on
// ties; where the spilling table pays (spill_pays), the global slab has to
// hold more than a third more of them.
// fixed_slab: visited slabs for a placement outside LDS, holding at most
// fixed_routes routes (the no-alloc entry point); nullptr: context scratch.
template <int kC, int kElem, int kR>
int launch_exact(Context* ctx, ExactArgs& a, int hash_mode, uint32_t lds_full,
                 uint32_t lds_spill, uint32_t lds_glob, uint32_t count, uint32_t* fixed_slab,
                 uint32_t fixed_routes)
{
    const int rf = exact_resident<kVisitedLds, kC, kElem, kR>(ctx, lds_full);
    const int rs = exact_resident<kVisitedSpill, kC, kElem, kR>(ctx, lds_spill);
    const int rg = exact_resident<kVisitedGlobal, kC, kElem, kR>(ctx, lds_glob);
    int mode = kVisitedLds;
    int res = rf;
    if (hash_mode == GOFANN_PLACE_GLOBAL) {
        mode = kVisitedGlobal;
        res = rg;
    } else if (hash_mode == GOFANN_PLACE_SPILL) {
        mode = kVisitedSpill;
        res = rs;
    } else if (hash_mode == GOFANN_PLACE_AUTO) {
        if (!full_table(ctx, count, lds_full, rf)) {
            if (rs > res) {
                mode = kVisitedSpill;
                res = rs;
            }
            if (rg > res + (spill_pays<kElem>(ctx, a, count, rs, rg) ? res / 3 : 0)) {
                mode = kVisitedGlobal;
                res = rg;
            }
        }
    }
    if (res <= 0)
        return ctx->fail(GOFANN_ERR_UNSUPPORTED, "per-route LDS state exceeds the workgroup limit");
    a.hash_global = nullptr;
    if (mode != kVisitedLds && fixed_slab != nullptr) {
        if (count > fixed_routes)
            return ctx->fail(GOFANN_ERR_INVALID,
                             "no-alloc exact search: " + std::to_string(count) +
                                 " routes need visited slabs beyond the fixed scratch (at most " +
                                 std::to_string(fixed_routes) +
                                 " routes per call with a visited set outside LDS)");
        a.hash_global = fixed_slab;
    } else if (mode != kVisitedLds) {
        const size_t need = static_cast<size_t>(count) * kHashCapacity * sizeof(uint32_t);
        a.hash_global = static_cast<uint32_t*>(ctx->scratch(Context::kScratchHash, need));
        if (!a.hash_global) return ctx->fail(GOFANN_ERR_NOMEM, "visited set scratch");
    }
    const uint32_t lds = mode == kVisitedLds ? lds_full : (mode == kVisitedSpill ? lds_spill : lds_glob);
    const dim3 grid(count), block(kWave);
    if (mode == kVisitedLds)
        hipLaunchKernelGGL((exact_kernel<kVisitedLds, kC, kElem, kR>()), grid, block, lds,
                           ctx->stream, a);
    else if (mode == kVisitedSpill)
        hipLaunchKernelGGL((exact_kernel<kVisitedSpill, kC, kElem, kR>()), grid, block, lds,
                           ctx->stream, a);
    else
        hipLaunchKernelGGL((exact_kernel<kVisitedGlobal, kC, kElem, kR>()), grid, block, lds,
                           ctx->stream, a);
    if (hipGetLastError() != hipSuccess) return ctx->fail_hip("exact route launch");
    ctx->last_table_in_lds = 0;
    ctx->last_hash_in_lds = mode == kVisitedGlobal ? 0 : (mode == kVisitedLds ? 1 : 2);
    ctx->last_lds_bytes = static_cast<int>(lds);
    ctx->last_resident = res;
    return GOFANN_OK;
}

// The set-frontier launches, defined in exact_set_*.hip.
#define GOFANN_EXACT_LAUNCH_ARGS                                                        \
    Context*, ExactArgs&, int, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t*, uint32_t
#define GOFANN_EXACT_SET_LAUNCHES(prefix, elem)                                         \
    prefix template int launch_exact<0, elem, 2>(GOFANN_EXACT_LAUNCH_ARGS);             \
    prefix template int launch_exact<0, elem, 4>(GOFANN_EXACT_LAUNCH_ARGS);             \
    prefix template int launch_exact<0, elem, 8>(GOFANN_EXACT_LAUNCH_ARGS);
#define GOFANN_EXACT_SET_LONG_LAUNCHES(prefix, elem)                                    \
    prefix template int launch_exact<-1, elem, 2>(GOFANN_EXACT_LAUNCH_ARGS);            \
    prefix template int launch_exact<-1, elem, 4>(GOFANN_EXACT_LAUNCH_ARGS);            \
    prefix template int launch_exact<-1, elem, 8>(GOFANN_EXACT_LAUNCH_ARGS);
extern template int launch_exact<0, GOFANN_ELEM_U8, 2>(GOFANN_EXACT_LAUNCH_ARGS);
GOFANN_EXACT_SET_LAUNCHES(extern, GOFANN_ELEM_F32)
GOFANN_EXACT_SET_LONG_LAUNCHES(extern, GOFANN_ELEM_F32)
GOFANN_EXACT_SET_LAUNCHES(extern, GOFANN_ELEM_F16)
GOFANN_EXACT_SET_LONG_LAUNCHES(extern, GOFANN_ELEM_F16)

}  // namespace gofann
