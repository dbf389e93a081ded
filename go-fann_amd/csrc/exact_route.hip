// exact_route.hip -- the full-GPU exact-distance route on gfx950.
//
// Reference: run_full_gpu_highfreq_route (src/search/full_gpu/
// backend_full_gpu.cu:1682-2042) launched by full_gpu_highfreq_kernel
// (:2045-2122).  A beam search whose frontier is keyed by the exact squared
// L2 distance (u8 vectors: l2_distance_device :1199-1244, an integer, here
// |b|^2 + |q|^2 - 2 b.q in u32 through v_dot4_u32_u8, converted to float;
// f32 and f16 vectors: :1107-1160, in that function's warp order, with the
// query in LDS as f32), with the route filter applied to every expanded
// node and a sorted best-k with sample dedup (insert_best_result
// :1342-1375).
//
// Per step (one wave64 per route):
//  * lane 0: filter of the expanded node (row mask & route bits, every active
//    legacy range, the route predicate when enabled) and its best-k insert;
//  * lane j: adjacency entry j of the node (prefetched at pickup), its
//    visited test, group bound and sample id, then (u8) the exact distance
//    of its own base row -- every lane streams a different row, 16 bytes a
//    load; float rows are scored in the reference's warp order, 16 at a
//    time (one per quad of lanes) or, past 4 KB a row, 2 at a time (one per
//    32-lane half) (exact_dist.hpp);
//  * candidates that cannot enter a full frontier are dropped in parallel,
//    the rest are admitted by lane 0 in adjacency order (smmh2 insert,
//    pop_max at Q+2), and the admitted rows enter the visited set;
//  * pickup of the next entry and the reference's early-stop rule (skipped on
//    the first transition): adaptive mode resets on an improved best-k,
//    otherwise a full best-k that the next entry cannot improve counts
//    towards early_stop_reached(mode, hits, finish, Q, expanded, passed, K).
//
// A route with no group rows, an invalid seed, or a seed sample past the
// base emits padding (UINT32_MAX / FLT_MAX) and zero steps.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>
#include <mutex>
#include <string>

#include "exact_route.hpp"

// Visited-set slabs of gofann_exact_search_noalloc: a fixed device array in
// place of context scratch, for callers that cannot allocate.  Each GPU the
// library runs on holds its own copy until the process ends.  Host code never
// passes this name to a kernel (on the host it is only a stand-in for the
// symbol); it uses the per-device address that hipGetSymbolAddress returned.
static __device__ __align__(256) uint32_t scratch[GOFANN_EXACT_NOALLOC_MAX_ROUTES * 4096u];

namespace gofann {

namespace {
constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mutex;
uint32_t* g_noalloc_slab[kNoAllocMaxDevices] = {};
std::string g_noalloc_error[kNoAllocMaxDevices];
}  // namespace

// Looks up this device's copy of `scratch` once (gofann_create calls it with
// the context's device current).  A failure is kept and reported by the
// no-alloc entry point; the other entry points do not need the array.
void noalloc_setup(int device)
{
    if (device < 0 || device >= kNoAllocMaxDevices) return;
    std::lock_guard<std::mutex> lock(g_noalloc_mutex);
    if (g_noalloc_slab[device] != nullptr) return;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
        (void)hipGetLastError();
        g_noalloc_error[device] = std::string("hipGetSymbolAddress(scratch): ") +
                                  hipGetErrorString(e);
        return;
    }
    g_noalloc_slab[device] = static_cast<uint32_t*>(p);
    g_noalloc_error[device].clear();
}

namespace {
inline uint32_t align16u(uint32_t x) { return (x + 15u) & ~15u; }
}  // namespace

struct LaunchShape {
    Context* ctx;
    ExactArgs* a;
    int hash_mode;
    uint32_t lds_full, lds_spill, lds_glob, count;
    uint32_t* fixed_slab;
    uint32_t fixed_routes;
};

// The heap-frontier kernels.  Row length fixed at compile time only in builds
// that ask for it (u8).
template <int kElem>
int launch_rows(const LaunchShape& s, int chunks)
{
    if constexpr (kElem != GOFANN_ELEM_U8) {
        if (chunks < 0)
            return launch_exact<-1, kElem, 0>(s.ctx, *s.a, s.hash_mode, s.lds_full, s.lds_spill,
                                              s.lds_glob, s.count, s.fixed_slab, s.fixed_routes);
    }
#if GOFANN_EXACT_FIXED_ROWS
    if constexpr (kElem == GOFANN_ELEM_U8) {
        switch (chunks) {
        case 8:
            return launch_exact<8, kElem, 0>(s.ctx, *s.a, s.hash_mode, s.lds_full, s.lds_spill,
                                             s.lds_glob, s.count, s.fixed_slab, s.fixed_routes);
        case 12:
            return launch_exact<12, kElem, 0>(s.ctx, *s.a, s.hash_mode, s.lds_full, s.lds_spill,
                                              s.lds_glob, s.count, s.fixed_slab, s.fixed_routes);
        case 16:
            return launch_exact<16, kElem, 0>(s.ctx, *s.a, s.hash_mode, s.lds_full, s.lds_spill,
                                              s.lds_glob, s.count, s.fixed_slab, s.fixed_routes);
        default:
            break;
        }
    }
#else
    (void)chunks;
#endif
    return launch_exact<0, kElem, 0>(s.ctx, *s.a, s.hash_mode, s.lds_full, s.lds_spill, s.lds_glob,
                                     s.count, s.fixed_slab, s.fixed_routes);
}

// The set-frontier kernels: R registers a lane hold the beam (set_registers).
template <int kElem, int kR>
int launch_set_r(const LaunchShape& s, int chunks)
{
    if constexpr (kElem != GOFANN_ELEM_U8) {
        if (chunks < 0)
            return launch_exact<-1, kElem, kR>(s.ctx, *s.a, s.hash_mode, s.lds_full, s.lds_spill,
                                               s.lds_glob, s.count, s.fixed_slab, s.fixed_routes);
    }
    return launch_exact<0, kElem, kR>(s.ctx, *s.a, s.hash_mode, s.lds_full, s.lds_spill, s.lds_glob,
                                      s.count, s.fixed_slab, s.fixed_routes);
}

template <int kElem>
int launch_set(const LaunchShape& s, int chunks, int regs)
{
    if constexpr (kElem == GOFANN_ELEM_U8) return launch_set_r<kElem, 2>(s, chunks);
    switch (regs) {
    case 2: return launch_set_r<kElem, 2>(s, chunks);
    case 4: return launch_set_r<kElem, 4>(s, chunks);
    default: return launch_set_r<kElem, 8>(s, chunks);
    }
}

static int exact_search_impl(Context* ctx, const void* base, int base_elem, uint32_t dim,
                             uint32_t samples, const void* queries, const gofann_graph_view* g,
                             const uint32_t* label_size, const gofann_predicate_view* pred,
                             const gofann_routes* r, const gofann_exact_params* p,
                             uint32_t* out_ids, float* out_dists, gofann_route_stats* stats,
                             uint32_t* fixed_slab, uint32_t fixed_routes)
{
    if (!g || !r || !p) return ctx->fail(GOFANN_ERR_INVALID, "null view");
    if (base_elem != GOFANN_ELEM_U8 && base_elem != GOFANN_ELEM_F32 && base_elem != GOFANN_ELEM_F16)
        return ctx->fail(GOFANN_ERR_INVALID, "base_elem must be u8, f32 or f16");
    if (!base || !queries || dim == 0)
        return ctx->fail(GOFANN_ERR_INVALID, "exact route vectors missing");
    if (dim > 65536) return ctx->fail(GOFANN_ERR_INVALID, "dim must be <= 65536 (u32 distances)");
    if (p->queue_limit < 2 || p->queue_limit > 1024)
        return ctx->fail(GOFANN_ERR_INVALID, "queue_limit must be in [2, 1024]");
    if (p->topk < 1 || p->topk > kExactMaxTopk)
        return ctx->fail(GOFANN_ERR_INVALID, "topk must be in [1, 10]");
    if (p->early_stop_mode < 0 || p->early_stop_mode > 2)
        return ctx->fail(GOFANN_ERR_INVALID, "unknown early stop mode");
    if (p->hash_mode < GOFANN_PLACE_AUTO || p->hash_mode > GOFANN_PLACE_SPILL)
        return ctx->fail(GOFANN_ERR_INVALID, "hash_mode in [0, 3]");
    if (!g->graph || !g->row_to_sample || !g->label_offset || g->degree == 0)
        return ctx->fail(GOFANN_ERR_INVALID, "graph view incomplete");
    if (g->degree > static_cast<uint32_t>(kMaxDegree))
        return ctx->fail(GOFANN_ERR_UNSUPPORTED, "graph degree must be in [1, 64]");
    if (r->count == 0) return GOFANN_OK;
    if (!r->route_query || !r->route_group || !r->route_start || !out_ids || !out_dists)
        return ctx->fail(GOFANN_ERR_INVALID, "route arrays or outputs missing");
    if ((reinterpret_cast<uintptr_t>(base) & 15u) != 0)
        return ctx->fail(GOFANN_ERR_INVALID, "base must be 16-byte aligned");

    ExactArgs a;
    a.graph = *g;
    a.label_size = label_size;
    a.pred = pred ? *pred : gofann_predicate_view{};
    a.routes = *r;
    a.base = static_cast<const uint8_t*>(base);
    a.queries = static_cast<const uint8_t*>(queries);
    a.dim = dim;
    a.samples = samples;
    a.params = *p;
    a.out_ids = out_ids;
    a.out_dists = out_dists;
    a.stats = stats;
    // LDS: the query row, then the frontier, then the visited table of the
    // chosen placement.
    a.off_frontier = base_elem == GOFANN_ELEM_U8 ? align16u((dim + 15u) / 16u * 16u)
                                                 : align16u(dim * 4u);
    a.off_heap = 0;
    a.log = nullptr;
    a.log_mask = 0;
    LaunchShape sh{ctx, &a, p->hash_mode, 0, 0, 0, r->count, fixed_slab, fixed_routes};
    const auto layout = [&](uint32_t frontier_bytes) {
        a.off_hash = align16u(a.off_frontier + frontier_bytes);
        sh.lds_full = a.off_hash + kHashCapacity * 4u;
        sh.lds_spill = a.off_hash + kSpillSlots * 4u;
        sh.lds_glob = a.off_hash;
    };
    // float rows over kQuadMaxRowBytes take the long-row kernel
    const int fchunks = static_cast<size_t>(dim) * elem_bytes(base_elem) > kQuadMaxRowBytes ? -1 : 0;
    const uint32_t q = static_cast<uint32_t>(p->queue_limit);
    // The set frontier serves float rows, whose distances are seldom equal
    // (4,900 f16 routes, dim 512: 9.9 ms, 10.5 with the heap), and u8 launches of
    // at most 16 routes and beams of at most two registers a lane (Q = 112).  A
    // u8 route that has equal keys which matter replays its admissions on the
    // heap, so the wider the beam and the more routes, the likelier is one that
    // takes longer than with the heap.  Set / heap, ms a launch at 1, 4, 16 and 32
    // routes: dim 192, degree 64, Q = 32: 0.25 / 0.35, 0.30 / 0.41, 0.34 / 0.46,
    // 0.37 / 0.48; Q = 112: 0.74 / 0.85, 0.89 / 0.94, 1.01 / 1.05, 1.10 / 1.10; Q =
    // 128: 0.88 / 0.94, 1.06 / 1.03, 1.23 / 1.16, 1.33 / 1.21; dim 32, degree 32,
    // Q = 72: 0.40 / 0.48, 0.51 / 0.55, 0.56 / 0.57, 0.65 / 0.59.
    const bool set_pays = base_elem != GOFANN_ELEM_U8 || (r->count <= 16 && q + kSetSlack <= 128);
    if (const int regs = fixed_slab == nullptr && set_pays
                             ? set_registers(ctx, p->queue_limit, r->count, &a.log) : 0) {
        a.log_mask = set_log_entries(p->queue_limit) - 1u;
        a.off_heap = align16u(a.off_frontier + set_capacity(p->queue_limit, regs) * 8u);
        layout(a.off_heap - a.off_frontier + split_heap_bytes(p->queue_limit));
        int rc;
        switch (base_elem) {
        case GOFANN_ELEM_F32: rc = launch_set<GOFANN_ELEM_F32>(sh, fchunks, regs); break;
        case GOFANN_ELEM_F16: rc = launch_set<GOFANN_ELEM_F16>(sh, fchunks, regs); break;
        default: rc = launch_set<GOFANN_ELEM_U8>(sh, 0, regs); break;
        }
        // The heap frontier runs where the set takes more LDS than a workgroup
        // has (below 64 slots it takes more than the heap) or where its rings
        // leave no memory for the visited slabs.
        if (rc != GOFANN_ERR_UNSUPPORTED && rc != GOFANN_ERR_NOMEM) return rc;
        if (rc == GOFANN_ERR_NOMEM) ctx->release(Context::kScratchLog);
    }
    const int chunks = (GOFANN_EXACT_FIXED_ROWS && (dim == 128 || dim == 192 || dim == 256))
                           ? static_cast<int>(dim / 16)
                           : 0;
    layout((q + 2u) * static_cast<uint32_t>(sizeof(Entry)));
    switch (base_elem) {
    case GOFANN_ELEM_F32: return launch_rows<GOFANN_ELEM_F32>(sh, fchunks);
    case GOFANN_ELEM_F16: return launch_rows<GOFANN_ELEM_F16>(sh, fchunks);
    default: return launch_rows<GOFANN_ELEM_U8>(sh, chunks);
    }
}

int exact_search(Context* ctx, const void* base, int base_elem, uint32_t dim, uint32_t samples,
                 const void* queries, const gofann_graph_view* g, const uint32_t* label_size,
                 const gofann_predicate_view* pred, const gofann_routes* r,
                 const gofann_exact_params* p, uint32_t* out_ids, float* out_dists,
                 gofann_route_stats* stats)
{
    return exact_search_impl(ctx, base, base_elem, dim, samples, queries, g, label_size, pred, r,
                             p, out_ids, out_dists, stats, nullptr, 0);
}

int exact_search_noalloc(Context* ctx, const void* base, int base_elem, uint32_t dim,
                         uint32_t samples, const void* queries, const gofann_graph_view* g,
                         const uint32_t* label_size, const gofann_predicate_view* pred,
                         const gofann_routes* r, const gofann_exact_params* p,
                         uint32_t* out_ids, float* out_dists, gofann_route_stats* stats)
{
    uint32_t* slab = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_noalloc_mutex);
        if (ctx->device >= 0 && ctx->device < kNoAllocMaxDevices)
            slab = g_noalloc_slab[ctx->device];
        if (slab == nullptr)
            return ctx->fail(GOFANN_ERR_HIP,
                             "no-alloc scratch unavailable on this device" +
                                 (ctx->device >= 0 && ctx->device < kNoAllocMaxDevices &&
                                          !g_noalloc_error[ctx->device].empty()
                                      ? ": " + g_noalloc_error[ctx->device]
                                      : std::string()));
    }
    return exact_search_impl(ctx, base, base_elem, dim, samples, queries, g, label_size, pred, r,
                             p, out_ids, out_dists, stats, slab, GOFANN_EXACT_NOALLOC_MAX_ROUTES);
}

}  // namespace gofann
