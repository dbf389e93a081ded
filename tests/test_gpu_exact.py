"""GPU parity of the full-GPU exact route (gofann_exact_search): ids,
distance bits and the eight per-route counters identical to the oracle,
across visited-set placements, neighbour-sample tables, early-stop modes,
beam sizes, route predicates and legacy bit/range filters, and every
distance path (u8 rows of fixed length 128/192/256, dim % 16 == 0, dim % 4
== 0, any dim; f32 and f16 rows in the warp order); and the exact posting
scans in both summation orders."""
from __future__ import annotations

import dataclasses
import sys

import numpy as np
import pytest
import torch

import pyoracle as po
from gofann_amd import _lib
from gofann_amd import index as gi
from gofann_amd import plan as gp
from gofann_amd import search as gs
from gofann_amd import synth

pytestmark = pytest.mark.gpu
U32MAX = 0xFFFFFFFF


def say(*a):
    print("[gpu-test]", *a, flush=True)
    sys.stdout.flush()


def _world(dim, seed, n=5000, nq=40):
    wl = synth.small_labelled(n=n, nq=nq, dim=dim, k=10, sigma=0.7, labels=5, seed=seed, tags=True,
                              dtype="u8")
    li = gi.build_label_index(wl.base, wl.label_offsets, wl.label_values, wl.num_labels,
                              wl.centroids, degree=32, threshold=300)
    pl = gp.plan_queries(li, wl.query_labels)
    return wl, li, pl.graph


@pytest.fixture(scope="module")
def eworld(gpu_ctx):
    return _world(128, 51)


ELEM = {np.dtype(np.uint8): _lib.ELEM_U8, np.dtype(np.float32): _lib.ELEM_F32,
        np.dtype(np.float16): _lib.ELEM_F16}


def _run(ctx, wl, li, rs, pred_o, pred_g, Q, topk, mode, hash_mode, nsamp, max_steps=0,
         finish=1, legacy=None, rows=None):
    base, q = rows if rows is not None else (wl.base.numpy(), wl.queries.numpy())
    kw = {}
    if legacy is not None:
        kw = dict(row_filter_mask=legacy["rmask"], query_filter_bits=legacy["qbits"],
                  range_modes=legacy["modes"], range_lower=legacy["lo"], range_upper=legacy["hi"],
                  base_range_values=legacy["brv"])
    oi, od, ost = po.exact_search(li, rs, pred_o, base, q, queue_limit=Q, topk=topk,
                                  early_stop_mode=mode, finish_limit=finish, max_steps=max_steps,
                                  label_size=li.label_size, **kw)
    dg = gs.DeviceGraph.upload(li, neighbor_samples=nsamp)
    dr = gs.DeviceRoutes.upload(rs)
    dev = dict(base=torch.from_numpy(np.ascontiguousarray(base)).cuda(),
               q=torch.from_numpy(np.ascontiguousarray(q)).cuda(), ls=gs.u32(li.label_size))
    rv = dr.routes_view()
    if legacy is not None:
        for k in ("rmask", "qbits"):
            dev[k] = torch.from_numpy(legacy[k].view(np.int64)).cuda()
        dev["modes"] = torch.from_numpy(legacy["modes"]).cuda()
        dev["lo"] = torch.from_numpy(legacy["lo"]).cuda()
        dev["hi"] = torch.from_numpy(legacy["hi"]).cuda()
        dev["brv"] = torch.from_numpy(legacy["brv"]).cuda()
        rv.row_filter_mask, rv.query_filter_bits = _lib.ptr(dev["rmask"]), _lib.ptr(dev["qbits"])
        rv.range_modes, rv.range_lower = _lib.ptr(dev["modes"]), _lib.ptr(dev["lo"])
        rv.range_upper, rv.base_range_values = _lib.ptr(dev["hi"]), _lib.ptr(dev["brv"])
        rv.range_count = legacy["modes"].shape[1]
    n = rs.count
    ids = torch.empty(n * topk, dtype=torch.int32, device="cuda")
    dists = torch.empty(n * topk, device="cuda")
    st = torch.zeros(n * 8, dtype=torch.int32, device="cuda")
    prm = _lib.ExactParams(Q, finish, mode, max_steps, topk, hash_mode)
    ctx.check(ctx.lib.gofann_exact_search(ctx.handle, _lib.ptr(dev["base"]), ELEM[base.dtype], wl.dim,
                                          wl.n, _lib.ptr(dev["q"]), dg.view(), _lib.ptr(dev["ls"]),
                                          pred_g(dr, dg), rv, prm, _lib.ptr(ids), _lib.ptr(dists),
                                          _lib.ptr(st)))
    torch.cuda.synchronize()
    assert np.array_equal(ids.cpu().numpy().view(np.uint32).reshape(n, topk), oi)
    assert np.array_equal(dists.cpu().numpy().reshape(n, topk).view(np.uint32), od.view(np.uint32))
    assert np.array_equal(st.cpu().numpy().reshape(n, 8), ost)
    return oi, ost


PLACE = {"auto": (_lib.PLACE_AUTO, False), "lds-nsamp": (_lib.PLACE_LDS, True),
         "global": (_lib.PLACE_GLOBAL, False), "spill-nsamp": (_lib.PLACE_SPILL, True)}


@pytest.mark.parametrize("place", list(PLACE))
# Beams up to 510 admit through the wave-parallel heap operations on the
# LDS frontier; past 512 slots (Q = 600) admission takes the serial lane-0
# sifts.
@pytest.mark.parametrize("mode,Q", [(2, 32), (0, 62), (2, 64), (2, 80), (1, 128), (2, 300),
                                    (2, 600)])
@pytest.mark.parametrize("with_pred", [False, True])
def test_exact_search_matches_oracle(gpu_ctx, eworld, place, mode, Q, with_pred):
    wl, li, rs = eworld
    hash_mode, nsamp = PLACE[place]
    say("exact search", place, "mode", mode, "Q", Q, "pred", with_pred)
    pred_o = po.PredicateArrays.from_plan(rs.predicate, li) if with_pred else None

    def pred_g(dr, dg):
        return dr.predicate_view(dg, 0.0, False) if with_pred else _lib.PredicateView()

    oi, ost = _run(gpu_ctx, wl, li, rs, pred_o, pred_g, Q, 10, mode, hash_mode, nsamp,
                   max_steps=300 if mode == 1 else 0, finish=2)
    assert (oi[:, 0] != U32MAX).sum() > rs.count // 2
    assert ost[:, 0].max() > 5


@pytest.fixture(scope="module")
def c2_shape_world(gpu_ctx):
    """The C2 bench shape: dim 192 u8 (fixed 12-chunk rows), degree 64, tags,
    trained k-means buckets, medoid seeds."""
    wl = synth.small_labelled(n=9000, nq=48, dim=192, k=14, sigma=0.7, labels=6, seed=57,
                              tags=True, dtype="u8")
    cen = gi.train_kmeans(wl.base, 14, seed=57)
    li = gi.build_label_index(wl.base, wl.label_offsets, wl.label_values, wl.num_labels, cen,
                              degree=64, threshold=300)
    return wl, li, gp.plan_queries(li, wl.query_labels).graph


@pytest.mark.parametrize("place", list(PLACE))
@pytest.mark.parametrize("mode,Q", [(2, 32), (2, 62), (2, 96), (2, 126), (0, 128), (2, 300)])
def test_exact_search_degree64_c2_shape(gpu_ctx, c2_shape_world, place, mode, Q):
    """Degree 64: lanes 32..63 of load_node/keep, the 64-bit ballot
    compaction and admissions of more than 32 neighbours per step."""
    wl, li, rs = c2_shape_world
    hash_mode, nsamp = PLACE[place]
    say("exact search degree 64", place, "mode", mode, "Q", Q)
    pred_o = po.PredicateArrays.from_plan(rs.predicate, li)
    oi, ost = _run(gpu_ctx, wl, li, rs, pred_o, lambda dr, dg: dr.predicate_view(dg, 0.0, False),
                   Q, 10, mode, hash_mode, nsamp, finish=2)
    assert (li.graph[:, 32:] != U32MAX).any(1).mean() > 0.5
    assert ost[:, 6].max() > 32  # some step admitted more than 32 neighbours overall
    if Q > 260:  # some frontier grew past 260 slots: pairs 64.. have children
        assert ost[:, 6].max() > 300
    assert (oi[:, 0] != U32MAX).sum() > rs.count // 2


def test_exact_search_legacy_filters_and_topk1(gpu_ctx, eworld):
    wl, li, rs = eworld
    say("exact search legacy filters")
    rng = np.random.default_rng(9)
    rc = 2
    legacy = dict(rmask=rng.integers(1, 4, li.row_to_sample.shape[0]).astype(np.uint64),
                  qbits=rng.integers(1, 4, rs.count).astype(np.uint64),
                  modes=rng.integers(0, 4, (rs.count, rc)).astype(np.uint8),
                  brv=rng.integers(0, 20, (wl.n, rc)).astype(np.float32))
    legacy["lo"] = rng.integers(0, 8, (rs.count, rc)).astype(np.float32)
    legacy["hi"] = legacy["lo"] + rng.integers(4, 12, (rs.count, rc)).astype(np.float32)
    for topk in (1, 10):
        _run(gpu_ctx, wl, li, rs, None, lambda dr, dg: _lib.PredicateView(), 48, topk, 2,
             _lib.PLACE_AUTO, True, legacy=legacy)


@pytest.mark.parametrize("dim", [44, 45, 48, 192, 256])
def test_exact_search_distance_paths(gpu_ctx, dim):
    wl, li, rs = _world(dim, 60 + dim, n=3000, nq=24)
    say("exact search dim", dim)
    _run(gpu_ctx, wl, li, rs, None, lambda dr, dg: _lib.PredicateView(), 32, 10, 2,
         _lib.PLACE_AUTO, False)


@pytest.mark.parametrize("overflow", [0, 3])
def test_exact_search_label_slab(gpu_ctx, eworld, overflow):
    """The route predicate reading each node's labels from a 16-byte slab in
    per-sample records (fetched with the adjacency row at pickup) in place
    of the CSR: results identical to the oracle's; overflow 3 sends every
    third row through the CSR."""
    wl, li, rs = eworld
    say("exact search label slab overflow", overflow)
    rec = gs.SampleRecords.build(torch.zeros(wl.n, 16, dtype=torch.uint8), li.csr_offsets,
                                 li.csr_labels, overflow_every=overflow)
    pred_o = po.PredicateArrays.from_plan(rs.predicate, li)
    for place, mode, Q in (("auto", 2, 48), ("spill-nsamp", 2, 96)):
        hash_mode, nsamp = PLACE[place]
        _run(gpu_ctx, wl, li, rs, pred_o,
             lambda dr, dg: dr.predicate_view(dg, 0.0, False, records=rec), Q, 10, mode,
             hash_mode, nsamp, finish=2)


def _float_world(dim, seed, n=4000, nq=32):
    wl = synth.small_labelled(n=n, nq=nq, dim=dim, k=10, sigma=0.7, labels=5, seed=seed,
                              tags=True)
    li = gi.build_label_index(wl.base, wl.label_offsets, wl.label_values, wl.num_labels,
                              wl.centroids, degree=32, threshold=300)
    return wl, li, gp.plan_queries(li, wl.query_labels).graph


@pytest.mark.parametrize("dim", [37, 100, 128, 512, 1031, 2049, 4096])
@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_exact_search_float_rows(gpu_ctx, dim, dtype):
    """f32 and f16 rows (and queries of the same type): distances in the
    reference's warp order, bit-identical to the oracle, with every
    visited-set placement; odd dim takes the per-element f16 path, 100
    leaves partials of unequal length.  Rows over 4 KB (f32 1031 and up,
    f16 2049 and up; 4096 is C3's shape) take the long-row kernel, whose
    lanes load 32 row words at a time: 1031 and 2049 leave a tail shorter
    than one such batch."""
    wl, li, rs = _float_world(dim, 70 + dim)
    t = np.float16 if dtype == "f16" else np.float32
    rows = (wl.base.numpy().astype(t), wl.queries.numpy().astype(t))
    pred_o = po.PredicateArrays.from_plan(rs.predicate, li)
    for place, mode, Q, with_pred in (("auto", 2, 32, False), ("lds-nsamp", 2, 80, True),
                                      ("global", 0, 128, False), ("spill-nsamp", 2, 300, True)):
        hash_mode, nsamp = PLACE[place]
        say("exact search float rows", dtype, "dim", dim, place, "Q", Q, "pred", with_pred)

        def pred_g(dr, dg):
            return dr.predicate_view(dg, 0.0, False) if with_pred else _lib.PredicateView()

        oi, ost = _run(gpu_ctx, wl, li, rs, pred_o if with_pred else None, pred_g, Q, 10, mode,
                       hash_mode, nsamp, finish=2, rows=rows)
        assert (oi[:, 0] != U32MAX).sum() > rs.count // 2
        assert ost[:, 0].max() > 5


@pytest.fixture(scope="module")
def scan_worlds(gpu_ctx):
    out = {}
    for dim in (37, 128, 512, 4096):
        wl = synth.small_labelled(n=6000, nq=24, dim=dim, k=10, sigma=0.7, labels=5,
                                  seed=90 + dim, tags=True)
        li = gi.build_label_index(wl.base, wl.label_offsets, wl.label_values, wl.num_labels,
                                  wl.centroids, degree=16, threshold=300)
        out[dim] = (wl, li)
    return out


def _scan_lists(rng, n, routes):
    """Posting lists with duplicates, UINT32_MAX, ids past the base, an
    empty list and lists longer than one LDS chunk."""
    sizes = rng.integers(0, 700, routes).astype(np.uint32)
    sizes[0] = 0
    sizes[1] = 5000
    sizes[2] = 2048
    offs = np.zeros(routes, np.uint32)
    offs[1:] = np.cumsum(sizes)[:-1]
    ids = rng.integers(0, n, int(sizes.sum())).astype(np.uint32)
    ids[offs[1] + 3000: offs[1] + 3100] = ids[offs[1]: offs[1] + 100]
    ids[rng.integers(0, len(ids), len(ids) // 20)] = U32MAX
    ids[rng.integers(0, len(ids), len(ids) // 20)] = n + 3
    return ids, offs, sizes


@pytest.mark.parametrize("dim", [37, 128, 512, 4096])
@pytest.mark.parametrize("dtype", ["u8", "f32", "f16"])
@pytest.mark.parametrize("order", [_lib.EXACT_ORDER_SERIAL, _lib.EXACT_ORDER_WARP])
def test_exact_posting_scan_matches_oracle(gpu_ctx, scan_worlds, dim, dtype, order):
    """gofann_exact_posting_scan: ids, distance bits and pass counts equal
    the oracle's in both summation orders, with and without the route
    predicate, for topk 1, 10 and 64.  Row lengths cover the serial order's
    LDS tiles (rows of 16-byte multiples, 4096 at the C3 shape) and its
    thread-per-row path (dim 37), and the warp order's unaligned blocks."""
    wl, li = scan_worlds[dim]
    x, qx = wl.base.numpy(), wl.queries.numpy()
    if dtype == "u8":
        lo, hi = float(x.min()), float(x.max())
        base = np.clip(np.round((x - lo) * 255.0 / (hi - lo)), 0, 255).astype(np.uint8)
        q = np.clip(np.round((qx - lo) * 255.0 / (hi - lo)), 0, 255).astype(np.uint8)
    else:
        t = np.float16 if dtype == "f16" else np.float32
        base, q = x.astype(t), qx.astype(t)
    rows = [(qi, ls[0], list(ls), []) for qi, ls in enumerate(wl.query_labels)]
    rs = gp._routeset(rows, li)
    rng = np.random.default_rng(dim + order)
    ids, offs, sizes = _scan_lists(rng, base.shape[0], rs.count)
    dg = gs.DeviceGraph.upload(li)
    dr = gs.DeviceRoutes.upload(rs)
    db = torch.from_numpy(base).cuda()
    dq = torch.from_numpy(q).cuda()
    for with_pred in (False, True):
        pred_o = po.PredicateArrays.from_plan(rs.predicate, li) if with_pred else None
        pv = dr.predicate_view(dg, 0.0, False) if with_pred else None
        for k in (1, 10, 64):
            say("exact posting scan", dtype, "dim", dim, "order", order, "pred", with_pred, "k", k)
            oi, od, op = po.exact_posting_scan(pred_o, base, q, rs.route_query, ids, offs, sizes,
                                               k, order)
            gi_, gd, gp_ = gs.exact_posting(gpu_ctx, db, dq, rs.route_query, ids, offs, sizes, k,
                                            order, pv)
            torch.cuda.synchronize()
            assert np.array_equal(gi_.cpu().numpy().view(np.uint32).reshape(-1, k), oi)
            assert np.array_equal(gd.cpu().numpy().reshape(-1, k).view(np.uint32),
                                  od.view(np.uint32))
            assert np.array_equal(gp_.cpu().numpy().view(np.uint32), op)
            assert (oi[:, 0] != U32MAX).sum() > rs.count // 2


@pytest.mark.parametrize("dtype,order", [("u8", _lib.EXACT_ORDER_SERIAL),
                                         ("f32", _lib.EXACT_ORDER_WARP)])
def test_exact_posting_scan_split_lists(gpu_ctx, scan_worlds, dtype, order):
    """Few routes: each list is cut into runs of whole 256-row passes that
    are merged.  List lengths at the edges of a run and of the number of
    runs, samples listed in several runs, no candidate in some runs."""
    dim = 37
    wl, li = scan_worlds[dim]
    x = wl.base.numpy()
    scale = 255.0 / float(x.max() - x.min())
    rows = lambda t: (np.clip(np.round((t - x.min()) * scale), 0, 255).astype(np.uint8)
                      if dtype == "u8" else t.astype(np.float32))
    base, q = rows(x), rows(wl.queries.numpy())
    sizes = np.array([0, 1, 255, 256, 257, 511, 512, 4095, 4096, 4097, 8191, 9000], np.uint32)
    offs = np.zeros(len(sizes), np.uint32)
    offs[1:] = np.cumsum(sizes)[:-1]
    rng = np.random.default_rng(5)
    ids = rng.integers(0, base.shape[0], int(sizes.sum())).astype(np.uint32)
    ids[offs[9]: offs[9] + 4097] = np.arange(4097) % 300     # every run lists the same samples
    ids[offs[10]: offs[10] + 4096] = U32MAX                  # runs without a candidate
    ids[offs[11]: offs[11] + 9000] = np.arange(9000) % 3     # fewer samples than k
    rq = np.arange(len(sizes), dtype=np.uint32)
    db, dq = torch.from_numpy(base).cuda(), torch.from_numpy(q).cuda()
    for k in (1, 10, 64):
        say("exact posting scan split lists", dtype, "order", order, "k", k)
        oi, od, op = po.exact_posting_scan(None, base, q, rq, ids, offs, sizes, k, order)
        gi_, gd, gp_ = gs.exact_posting(gpu_ctx, db, dq, rq, ids, offs, sizes, k, order, None)
        torch.cuda.synchronize()
        assert np.array_equal(gi_.cpu().numpy().view(np.uint32).reshape(-1, k), oi)
        assert np.array_equal(gd.cpu().numpy().reshape(-1, k).view(np.uint32), od.view(np.uint32))
        assert np.array_equal(gp_.cpu().numpy().view(np.uint32), op)


def test_exact_search_invalid_seeds(gpu_ctx, eworld):
    wl, li, rs = eworld
    say("exact search invalid seeds")
    start = rs.route_start.copy()
    start[0] = U32MAX
    start[1] = li.label_size[rs.route_group[1]]
    rs2 = gp.RouteSet(rs.route_query, rs.route_group, start, rs.route_to_query, rs.predicate)
    oi, ost = _run(gpu_ctx, wl, li, rs2, None, lambda dr, dg: _lib.PredicateView(), 32, 10, 2,
                   _lib.PLACE_AUTO, False)
    assert np.all(oi[:2] == U32MAX) and np.all(ost[:2, 0] == 0)


def test_exact_search_rejects_bad_params(gpu_ctx, eworld):
    wl, li, rs = eworld
    dg = gs.DeviceGraph.upload(li)
    dr = gs.DeviceRoutes.upload(rs)
    base, q = wl.base.cuda(), wl.queries.cuda()
    for Q, k, elem in ((1, 10, _lib.ELEM_U8), (32, 11, _lib.ELEM_U8), (32, 10, 3)):
        prm = _lib.ExactParams(Q, 1, 2, 0, k, 0)
        rc = gpu_ctx.lib.gofann_exact_search(gpu_ctx.handle, _lib.ptr(base), elem, wl.dim, wl.n,
                                             _lib.ptr(q), dg.view(), None, _lib.PredicateView(),
                                             dr.routes_view(), prm, None, None, None)
        assert rc in (_lib.ERR_INVALID, _lib.ERR_UNSUPPORTED)


# ---- the set frontier (set_frontier.hpp), which float launches take, and u8
# launches of at most 16 routes and beams up to 112
def _sixteens(rs):
    """The routes sixteen at a time, then the heap's seventeen."""
    for a, b in [(a, min(rs.count, a + 16)) for a in range(0, rs.count, 16)] + [(0, 17)]:
        yield dataclasses.replace(rs, route_query=rs.route_query[a:b],
                                  route_group=rs.route_group[a:b],
                                  route_start=rs.route_start[a:b],
                                  route_to_query=rs.route_to_query[a:b])


@pytest.mark.parametrize("shift", [4, 6, 7])
@pytest.mark.parametrize("Q", [2, 7, 48, 111, 112, 113, 240, 241, 496, 497])
def test_exact_search_equal_distances(gpu_ctx, eworld, shift, Q):
    """Rows of 16, 4 and 2 distinct values a dim: many equal distances, so
    that the order of the heap decides who is next and who leaves.  The set
    frontier serves the u8 beams up to 112, the heap those past it."""
    wl, li, rs = eworld
    say("exact search, equal distances", shift, "Q", Q)
    rows = (wl.base.numpy()[:, :12] >> shift, wl.queries.numpy()[:, :12] >> shift)
    rows = tuple(np.ascontiguousarray(r) for r in rows)

    class Small:
        dim, n = 12, wl.n
        base, queries = wl.base, wl.queries
    for part in _sixteens(rs):
        _run(gpu_ctx, Small, li, part, None, lambda dr, dg: _lib.PredicateView(), Q, 10, 2,
             _lib.PLACE_AUTO, False, rows=rows)


@pytest.mark.parametrize("Q", [2, 111, 112, 113, 240, 241, 496, 497])
@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_exact_search_equal_float_distances(gpu_ctx, eworld, dtype, Q):
    """The same for float rows, which take the set frontier whatever the
    number of routes: integer rows of 4 distinct values a dim (their sums are
    exact in either type).  112, 240 and 496 are the last beams of two, four
    and eight registers a lane; 497 takes the heap."""
    wl, li, rs = eworld
    say("exact search, equal float distances", dtype, "Q", Q)
    dt = np.float32 if dtype == "f32" else np.float16
    rows = tuple(np.ascontiguousarray((r.numpy()[:, :12] >> 6).astype(dt))
                 for r in (wl.base, wl.queries))

    class Small:
        dim, n = 12, wl.n
    _run(gpu_ctx, Small, li, rs, None, lambda dr, dg: _lib.PredicateView(), Q, 10, 2,
         _lib.PLACE_AUTO, False, rows=rows)


def _run_both(ctx, li, rs, base, q, Q, mode):
    """gofann_exact_search (set frontier) and gofann_exact_search_noalloc
    (heap frontier) on the same inputs."""
    dg, dr = gs.DeviceGraph.upload(li), gs.DeviceRoutes.upload(rs)
    b, qd = torch.from_numpy(base).cuda(), torch.from_numpy(q).cuda()
    ls = gs.u32(li.label_size)
    out = []
    for fn in (ctx.lib.gofann_exact_search, ctx.lib.gofann_exact_search_noalloc):
        n = rs.count
        ids = torch.empty(n * 10, dtype=torch.int32, device="cuda")
        dists = torch.empty(n * 10, device="cuda")
        st = torch.zeros(n * 8, dtype=torch.int32, device="cuda")
        prm = _lib.ExactParams(Q, 1, mode, 0, 10, _lib.PLACE_AUTO)
        ctx.check(fn(ctx.handle, _lib.ptr(b), ELEM[base.dtype], base.shape[1], base.shape[0],
                     _lib.ptr(qd), dg.view(), _lib.ptr(ls), _lib.PredicateView(),
                     dr.routes_view(), prm, _lib.ptr(ids), _lib.ptr(dists), _lib.ptr(st)))
        torch.cuda.synchronize()
        out.append([ids.cpu().numpy(), dists.cpu().numpy().view(np.uint32), st.cpu().numpy()])
    return out


@pytest.mark.parametrize("Q", [8, 96, 200, 448])
@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("kind", ["nan", "inf", "zero", "huge"])
def test_exact_search_unordered_distances(gpu_ctx, eworld, dtype, Q, kind):
    """NaN, infinite, all-zero and overflowing distances: the set frontier
    gives what the heap frontier gives."""
    wl, li, rs = eworld
    say("exact search", kind, dtype, "Q", Q)
    rng = np.random.default_rng(Q)
    base = (rng.standard_normal((wl.n, 24))).astype(np.float32)
    q = (rng.standard_normal((wl.queries.shape[0], 24))).astype(np.float32)
    hit = rng.random(wl.n) < 0.1
    if kind == "nan":
        base[hit, 3] = np.nan
        base[rng.random(wl.n) < 0.02, 5] = -np.nan
    elif kind == "inf":
        base[hit, 3] = np.inf
        base[rng.random(wl.n) < 0.1, 5] = -np.inf
        q[::3, 3] = np.inf
    elif kind == "zero":
        base[:] = 0
        q[::2] = 0
    else:
        base[hit] *= 1e20 if dtype == "f32" else 1e4
    dt = np.float32 if dtype == "f32" else np.float16
    with np.errstate(over="ignore"):
        base, q = base.astype(dt), q.astype(dt)
    for part in _sixteens(rs):
        a, b = _run_both(gpu_ctx, li, part, base, q, Q, 2)
        for x, y in zip(a, b):
            assert np.array_equal(x, y)


def test_exact_search_without_early_stop(gpu_ctx, eworld):
    """Whole routes: the set frontier gives what the heap frontier gives."""
    wl, li, rs = eworld
    say("exact search, no early stop")
    rng = np.random.default_rng(3)
    base = rng.standard_normal((wl.n, 32)).astype(np.float32)
    q = rng.standard_normal((wl.queries.shape[0], 32)).astype(np.float32)
    for Q in (112, 496):
        for part in _sixteens(rs):
            a, b = _run_both(gpu_ctx, li, part, base, q, Q, 1)
            for x, y in zip(a, b):
                assert np.array_equal(x, y)


def _line_world(n, degree=32):
    """One group whose row i links to the next `degree` rows, each nearer to
    the queries than the last, the seed farthest: a search admits every row.
    The last 400 rows are four at each of 100 distances."""
    i = np.arange(n, dtype=np.int64)
    nxt = i[:, None] + 1 + np.arange(degree)[None, :]
    graph = np.where(nxt < n, nxt, U32MAX).astype(np.uint32)
    rows = i.astype(np.uint32)
    li = gi.LabelIndex(1, 0, np.array([n]), np.zeros(1, np.uint32), np.array([n], np.uint32), rows,
                       graph, np.zeros(1, np.uint32), np.array([0, n], np.uint64), rows,
                       np.arange(n + 1, dtype=np.uint32), np.zeros(n, np.uint32), degree)
    rs = gp._routeset([(q, 0, [], []) for q in range(6)], li)
    x = np.zeros((n, 8), np.float32)
    x[:, 0] = n - i
    x[-400:, 0] = np.repeat(np.arange(100, 0, -1), 4)
    q = np.zeros((6, 8), np.float32)
    q[:, 1] = np.arange(6)
    return li, rs, x, q


@pytest.mark.parametrize("Q,ring", [(2, 1024), (112, 1024), (113, 2048), (496, 2048)])
def test_exact_search_log_ring_wraps(gpu_ctx, Q, ring):
    """Routes that admit more than twice what the log ring holds, with no
    equal keys until the end: a full ring brings the heap up to date, and
    the order among the equal keys that follow depends on all of it."""
    say("exact search, log ring", Q)
    li, rs, x, q = _line_world(6000)

    class Line:
        dim, n = 8, 6000
    _, st = _run(gpu_ctx, Line, li, rs, None, lambda dr, dg: _lib.PredicateView(), Q, 10, 1,
                 _lib.PLACE_AUTO, False, rows=(x, q))
    assert st[:, 6].min() > 2 * ring


def test_exact_scan_beside_a_capture(gpu_ctx, scan_worlds):
    """A context's first scan, which allocates its part lists, while torch
    captures a graph on another stream: both complete."""
    wl, _ = scan_worlds[128]
    say("exact posting scan beside a capture")
    base, q = wl.base.float().cuda(), wl.queries.float().cuda()
    n = int(q.shape[0])
    ids = np.random.default_rng(8).integers(0, wl.n, n * 900).astype(np.uint32)
    offs, sizes = np.arange(n, dtype=np.uint32) * 900, np.full(n, 900, np.uint32)
    rq = np.arange(n, dtype=np.uint32)
    want = po.exact_posting_scan(None, wl.base.float().numpy(), wl.queries.float().numpy(), rq, ids,
                                 offs, sizes, 10, _lib.EXACT_ORDER_SERIAL)
    dev = [gs.u32(a) for a in (rq, ids, offs, sizes)]
    out = [torch.zeros(n * 10, dtype=torch.int32, device="cuda"), torch.zeros(n * 10, device="cuda"),
           torch.zeros(n, dtype=torch.int32, device="cuda")]
    ctx = _lib.Context(0)
    side, cap, graph = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    ctx.bind_stream(side)
    x = torch.zeros(64, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(cap):
        graph.capture_begin()
        x.add_(1.0)
        ctx.check(ctx.lib.gofann_exact_posting_scan(
            ctx.handle, _lib.ptr(base), _lib.ELEM_F32, 128, wl.n, _lib.ptr(q),
            _lib.PredicateView(), *[_lib.ptr(t) for t in dev], n, 10, _lib.EXACT_ORDER_SERIAL,
            *[_lib.ptr(t) for t in out]))
        graph.capture_end()
    side.synchronize()
    for step in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert x.cpu().tolist() == [step + 1.0] * 64
    assert np.array_equal(out[0].cpu().numpy().view(np.uint32).reshape(n, 10), want[0])
    assert np.array_equal(out[1].cpu().numpy().reshape(n, 10).view(np.uint32),
                          want[1].view(np.uint32))
    ctx.close()


def test_exact_searches_beside_a_scan(gpu_ctx, eworld, scan_worlds):
    """Two contexts on streams of their own, searches on one beside scans on
    the other, alternating batch sizes: each gives what it gives alone."""
    wl, li, rs = eworld
    say("exact searches beside a scan")
    dg, dr = gs.DeviceGraph.upload(li), gs.DeviceRoutes.upload(rs)
    base, q = wl.base.float().cuda(), wl.queries.float().cuda()
    ls = gs.u32(li.label_size)
    n = int(q.shape[0])
    rng = np.random.default_rng(12)
    ids = rng.integers(0, wl.n, n * 900).astype(np.uint32)
    lists = [gs.u32(a) for a in (np.arange(n, dtype=np.uint32), ids,
                                 np.arange(n, dtype=np.uint32) * 900, np.full(n, 900, np.uint32))]

    def search(ctx, count, out):
        prm = _lib.ExactParams(96, 1, 2, 0, 10, _lib.PLACE_AUTO)
        ctx.check(ctx.lib.gofann_exact_search(
            ctx.handle, _lib.ptr(base), _lib.ELEM_F32, wl.dim, wl.n, _lib.ptr(q), dg.view(),
            _lib.ptr(ls), _lib.PredicateView(), dr.routes_view(0, count), prm, _lib.ptr(out[0]),
            _lib.ptr(out[1]), None))

    def scan(ctx, count, out):
        ctx.check(ctx.lib.gofann_exact_posting_scan(
            ctx.handle, _lib.ptr(base), _lib.ELEM_F32, wl.dim, wl.n, _lib.ptr(q),
            _lib.PredicateView(), *[_lib.ptr(t) for t in lists], count, 10,
            _lib.EXACT_ORDER_SERIAL, _lib.ptr(out[0]), _lib.ptr(out[1]), None))

    def buffers():
        return (torch.zeros(max(n, rs.count) * 10, dtype=torch.int32, device="cuda"),
                torch.zeros(max(n, rs.count) * 10, device="cuda"))

    counts = [(3, n), (rs.count, 5), (17, n), (rs.count, n)]
    want = []
    for a, b in counts:
        o = buffers(), buffers()
        search(gpu_ctx, a, o[0])
        scan(gpu_ctx, b, o[1])
        want.append(o)
    ctxs, streams = [_lib.Context(0) for _ in range(2)], [torch.cuda.Stream() for _ in range(2)]
    got = [(buffers(), buffers()) for _ in counts]
    torch.cuda.synchronize()
    for c, s in zip(ctxs, streams):
        c.bind_stream(s)
    for (a, b), o in zip(counts, got):
        search(ctxs[0], a, o[0])
        scan(ctxs[1], b, o[1])
    torch.cuda.synchronize()
    for w, g in zip(want, got):
        for x, y in zip(w, g):
            assert torch.equal(x[0], y[0])
            assert torch.equal(x[1].view(torch.int32), y[1].view(torch.int32))
    for c in ctxs:
        c.close()
