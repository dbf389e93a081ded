"""The work a user of this framework has it do, as cases to be timed: the
graph searches (exact, PQ, RaBitQ), the posting scans, and the construction
of graphs and codes, through the C ABI and its Python driver.

Every case is a dict of plain values.  `kind` picks the path:
  exact       gofann_exact_search over label graphs, then the route merge
  pq          gofann_pq_search, inline exact ranking or a shortlist that
              gofann_exact_rerank ranks, then the route merge
  rabitq      gofann_rabitq_prepare_queries, gofann_rabitq_search,
              gofann_exact_rerank, gofann_merge_routes: a whole batch
  range_scan  gofann_rabitq_range_scan_resident over narrow attribute ranges
  label_scan  gofann_rabitq_posting_scan_segments / _shared over label postings
  exact_scan  gofann_exact_posting_scan
  graph       index.build_label_index: label graphs from vectors and labels
  codes       the quantizers: PQ training and encoding, RaBitQ encoding

Vectors come from the mixtures of gofann_amd.synth (u8: centres uniform in
[32, 224]; floats: centre + low-rank spread + noise, normalised), labels are
Zipf(1.1), attributes uniform.
"""
from __future__ import annotations

import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "go-fann_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from gofann_amd import _lib  # noqa: E402
from gofann_amd import builder as gb  # noqa: E402
from gofann_amd import index as gi  # noqa: E402
from gofann_amd import plan as gp  # noqa: E402
from gofann_amd import range_posting as rp  # noqa: E402
from gofann_amd import search as gs  # noqa: E402

TOPK = 10
DEV = "cuda"
TORCH = {"u8": torch.uint8, "f16": torch.float16, "f32": torch.float32}
ELEM = {"u8": _lib.ELEM_U8, "f16": _lib.ELEM_F16, "f32": _lib.ELEM_F32}
SIZE = {"u8": 1, "f16": 2, "f32": 4}
ATTR = 10_000  # attribute values are integers in [0, ATTR)


def listed():
    return [
        # one query of an interactive user: latency, a single route on the chip
        dict(name="exact_u8_one", kind="exact", elem="u8", n=500_000, dim=192, degree=64,
             labels=8, filter="tags", queries=1, beam=64),
        # a server's micro-batch, far fewer routes than the chip holds
        dict(name="exact_u8_serve", kind="exact", elem="u8", n=1_000_000, dim=192, degree=64,
             labels=24, filter="tags", queries=200, beam=88),
        # the throughput batch of the benchmark's u8 workload
        dict(name="exact_u8_batch", kind="exact", elem="u8", n=3_000_000, dim=192, degree=64,
             labels=24, filter="tags", queries=40_000, beam=72),
        # f16 embeddings with label and interval filters, wide beam
        dict(name="exact_f16_batch", kind="exact", elem="f16", n=1_000_000, dim=512, degree=32,
             labels=24, filter="interval", queries=3_000, beam=416),
        # PQ codes with f32 rows, the beam ranked by exact distances inline
        dict(name="pq_f32_inline", kind="pq", elem="f32", n=1_000_000, dim=128, degree=32,
             labels=10, filter="tags", queries=6_000, beam=192, subspaces=32, inline=True),
        # one-bit codes over f16 embeddings: preparation, beam, rerank, merge
        dict(name="rabitq_f16_batch", kind="rabitq", elem="f16", n=2_000_000, dim=512, degree=32,
             labels=40, filter="interval", queries=8_000, beam=448, width=100, anchors=256),
        # one-bit codes over long f32 rows with half-open range filters
        dict(name="rabitq_f32_long", kind="rabitq", elem="f32", n=80_000, dim=4096, degree=32,
             labels=1, filter="range", queries=1_200, beam=320, width=200, anchors=128),
        # narrow ranges: every row of a slice of the attribute order
        dict(name="range_scan_long", kind="range_scan", n=120_000, dim=4096, routes=1_500,
             rows=4_000, width=200, anchors=128),
        # label postings with a residual label and range, many routes a label
        dict(name="label_scan_shared", kind="label_scan", n=500_000, dim=512, labels=60,
             routes=3_000, width=100, anchors=128),
        # narrow ranges by exact distances of f32 rows
        dict(name="exact_scan_f32", kind="exact_scan", elem="f32", n=120_000, dim=1024,
             routes=600, rows=4_000, order="serial"),
        # building: k-means buckets, kNN and links of every label's graph
        dict(name="graph_f16", kind="graph", elem="f16", n=150_000, dim=512, degree=32, labels=6,
             centres=256),
        # quantizing: PQ codebooks from a sample, then every row's codes
        dict(name="codes_pq_u8", kind="codes", codec="pq", elem="u8", n=1_000_000, dim=192,
             subspaces=48),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["exact", "exact", "exact", "pq", "rabitq", "rabitq", "range_scan",
                       "label_scan", "exact_scan", "graph", "codes"])
    if kind == "exact":
        elem = rng.choice(["u8", "u8", "f16", "f32"])
        dim = _log(rng, 24, 256) if elem == "u8" else _log(rng, 48, 640)
        if rng.random() < 0.5:
            dim = (dim + 15) // 16 * 16
        return dict(kind=kind, elem=elem, n=_log(rng, 20_000, 300_000), dim=dim,
                    degree=rng.choice([24, 32, 48, 64]), labels=rng.randint(2, 24),
                    filter="tags" if elem == "u8" else rng.choice(["tags", "interval"]),
                    queries=_log(rng, 1, 5_000 if elem == "u8" else 1_000),
                    beam=_log(rng, 16, 320))
    if kind == "pq":
        m = rng.choice([16, 24, 32, 48, 64])
        return dict(kind=kind, elem=rng.choice(["u8", "f32"]), n=_log(rng, 20_000, 300_000),
                    dim=4 * m, degree=rng.choice([32, 48, 64]), labels=rng.randint(2, 24),
                    filter="tags", queries=_log(rng, 1, 3_000), beam=_log(rng, 32, 192),
                    subspaces=m, inline=rng.random() < 0.5)
    if kind == "rabitq":
        elem = rng.choice(["f16", "f32"])
        dim = _log(rng, 100, 1024)
        return dict(kind=kind, elem=elem, n=_log(rng, 20_000, 300_000), dim=dim,
                    degree=rng.choice([24, 32, 64]), labels=rng.randint(2, 30),
                    filter=rng.choice(["interval", "range"]), queries=_log(rng, 1, 2_000),
                    beam=_log(rng, 16, 480), width=rng.choice([10, 50, 100, 200]),
                    anchors=rng.choice([64, 128, 256]))
    if kind == "range_scan":
        return dict(kind=kind, n=_log(rng, 20_000, 120_000), dim=128 * _log(rng, 1, 32),
                    routes=_log(rng, 1, 1_000), rows=_log(rng, 100, 4_000),
                    width=rng.choice([10, 100, 200]), anchors=rng.choice([64, 128]))
    if kind == "label_scan":
        return dict(kind=kind, n=_log(rng, 50_000, 500_000), dim=128 * rng.choice([1, 2, 4, 6, 8]),
                    labels=_log(rng, 10, 200), routes=_log(rng, 1, 2_000),
                    width=rng.choice([10, 50, 100]), anchors=rng.choice([64, 128]))
    if kind == "exact_scan":
        elem = rng.choice(["u8", "f16", "f32"])
        return dict(kind=kind, elem=elem, n=_log(rng, 20_000, 120_000), dim=_log(rng, 48, 1024),
                    routes=_log(rng, 1, 500), rows=_log(rng, 100, 4_000),
                    order=rng.choice(["serial", "warp"]))
    if kind == "graph":
        return dict(kind=kind, elem=rng.choice(["u8", "f16", "f32"]),
                    n=_log(rng, 20_000, 120_000), dim=_log(rng, 32, 400),
                    degree=rng.choice([24, 32, 64]), labels=rng.randint(1, 8),
                    centres=rng.choice([64, 128, 256]))
    if rng.random() < 0.5:
        m = rng.choice([16, 32, 48])
        return dict(kind=kind, codec="pq", elem=rng.choice(["u8", "f32"]),
                    n=_log(rng, 20_000, 300_000), dim=4 * m, subspaces=m)
    return dict(kind=kind, codec="rabitq", elem=rng.choice(["f16", "f32"]),
                n=_log(rng, 20_000, 200_000), dim=_log(rng, 100, 768), anchors=128)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed, role):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000 + role)
    return g


def _padded(dim):
    return (dim + 127) // 128 * 128


def _vectors(case, seed, nq):
    """Base rows and `nq` queries of one mixture; queries have the base's
    type, f32 for f16 rows."""
    n, dim, elem = case["n"], case["dim"], case.get("elem", "f32")
    k = max(8, min(256, n // 1500))
    g = _gen(seed, 1)
    if elem == "u8":
        cen = 32.0 + 192.0 * torch.rand(k, dim, generator=g, device=DEV)
    else:
        cen = torch.randn(k, dim, generator=g, device=DEV)
        basis = torch.randn(64, dim, generator=g, device=DEV)

    def rows(m, dtype, gen):
        cl = torch.randint(0, k, (m,), generator=gen, device=DEV)
        out = torch.empty(m, dim, dtype=dtype, device=DEV)
        step = max(1, (1 << 27) // dim)
        for s in range(0, m, step):
            e = min(m, s + step)
            noise = torch.randn(e - s, dim, generator=gen, device=DEV)
            if elem == "u8":
                x = (cen[cl[s:e]] + 16.0 * noise).round_().clamp_(0, 255)
            else:
                z = torch.randn(e - s, 64, generator=gen, device=DEV) * (0.7 / 8.0)
                x = cen[cl[s:e]] + z @ basis + 0.05 * noise
                x /= x.norm(dim=1, keepdim=True)
            out[s:e] = x.to(dtype)
        return out

    base = rows(n, TORCH[elem], _gen(seed, 2))
    queries = rows(nq, torch.uint8 if elem == "u8" else torch.float32, _gen(seed, 4))
    return base, queries


def _zipf(vocab):
    w = 1.0 / np.arange(1, vocab + 1, dtype=np.float64) ** 1.1
    return w / w.sum()


def _csr(rows, vocab):
    """Sorted CSR of an [n][k] label matrix; entries >= vocab and repeats drop."""
    rows = np.sort(rows, axis=1)
    keep = rows < vocab
    keep[:, 1:] &= rows[:, 1:] != rows[:, :-1]
    off = np.zeros(len(rows) + 1, np.uint32)
    np.cumsum(keep.sum(1), out=off[1:])
    return off, rows[keep].astype(np.uint32)


def _labels(case, rng):
    """(CSR offsets, labels, vocabulary, attribute [n][1] or None)."""
    n, vocab = case["n"], case["labels"]
    how = case["filter"]
    if how == "pairs":  # two distinct tags a row
        a = rng.choice(vocab, size=n, p=_zipf(vocab))
        b = (a + rng.integers(1, max(vocab, 2), size=n)) % vocab
        return *_csr(np.stack([a, b], 1), vocab), vocab, None
    if how == "tags":  # one to three tags a row
        m = rng.choice(vocab, size=(n, 3), p=_zipf(vocab))
        m[np.arange(3)[None, :] >= rng.integers(1, 4, size=n)[:, None]] = vocab
        return *_csr(m, vocab), vocab, None
    attr = rng.integers(0, ATTR, size=(n, 1)).astype(np.float32)
    if how == "range":
        return np.arange(n + 1, dtype=np.uint32), np.zeros(n, np.uint32), 1, attr
    cat = rng.choice(vocab, size=n, p=_zipf(vocab))  # a category and ten attribute intervals
    iv = vocab + (attr[:, 0].astype(np.int64) * 10 // ATTR)
    return *_csr(np.stack([cat, iv], 1), vocab + 10), vocab + 10, attr


def _routes(case, rng, li, nq):
    """Graph routes of the batch's filters, ordered by label group."""
    vocab = case["labels"]
    if case["filter"] == "tags":  # an AND of one or two tags
        a = rng.choice(vocab, size=(nq, 2), p=_zipf(vocab))
        two = (rng.random(nq) < 0.5) & (a[:, 0] != a[:, 1])
        ql = [sorted(r.tolist()) if t else [int(r[0])] for r, t in zip(a, two)]
        return gp.plan_queries(li, ql).graph
    wide = rng.uniform(0.05, 0.5 if case["filter"] == "range" else 0.2, size=nq)
    lo = np.floor(rng.random(nq) * (1.0 - wide) * ATTR)
    hi = np.floor(lo + wide * ATTR)
    rng_of = [(0, 3, float(a), float(b)) for a, b in zip(lo, hi)]
    if case["filter"] == "range":
        rows = [(q, 0, [], [rng_of[q]]) for q in range(nq)]
    else:  # half the queries by category, half by range over interval graphs
        cat = rng.choice(vocab, size=nq, p=_zipf(vocab))
        ql = [[int(cat[q])] if q % 2 == 0 else [] for q in range(nq)]
        qr = [[] if q % 2 == 0 else [rng_of[q]] for q in range(nq)]
        rows, _, _ = gp.interval_route_rows(li, ql, qr, vocab, 10, ATTR)
        rows = [r for r in rows if li.has_graph(r[1])]
    rows.sort(key=lambda r: (r[1], r[0]))
    return gp._routeset(rows, li)


def _orthogonal(P, seed):
    """[P][P] orthogonal matrix: a Kronecker product of two random ones with
    random column signs."""
    g = torch.Generator()
    g.manual_seed(int(seed) * 1000 + 5)
    a = torch.linalg.qr(torch.randn(P // 128, P // 128, generator=g))[0]
    b = torch.linalg.qr(torch.randn(128, 128, generator=g))[0]
    sign = torch.randint(0, 2, (P,), generator=g) * 2.0 - 1.0
    return (torch.kron(a, b) * sign[None, :]).to(DEV).contiguous()


def _graph_world(case, seed):
    """Index, routes and device views of a graph search."""
    rng = np.random.default_rng(seed * 1000 + 3)
    nq = case["queries"]
    base, queries = _vectors(case, seed, nq)
    off, lab, vocab, attr = _labels(case, rng)
    centres = gi.train_kmeans(base, max(8, min(128, case["n"] // 1500)), iters=3, sample=16384)
    li = gi.build_label_index(base, off, lab, vocab, centres, case["degree"], threshold=20)
    routes = _routes(case, rng, li, nq)
    st = dict(ctx=_lib.Context(0), base=base, queries=queries, n_routes=routes.count,
              dg=gs.DeviceGraph.upload(li, neighbor_samples=True),
              dr=gs.DeviceRoutes.upload(routes, attr), label_size=gs.u32(li.label_size),
              centres=centres, attr=attr, csr=(li.csr_offsets, li.csr_labels))
    q_off, q_routes = gs.query_route_csr(routes.route_query, nq)
    st["q_off"], st["q_routes"] = gs.u32(q_off), gs.u32(q_routes)
    st["ids"], st["dists"] = _route_rows(case, TOPK)
    return st


def _route_rows(case, width):
    """Output rows for as many routes as the batch's filters can have: two
    for an AND of two tags, three for a range over intervals."""
    n = case["queries"] * {"tags": 2, "interval": 3, "range": 1}[case["filter"]] * width
    return (torch.full((n,), -1, dtype=torch.int32, device=DEV),
            torch.zeros(n, dtype=torch.float32, device=DEV))


def _prepare_exact(case, seed):
    st = _graph_world(case, seed)
    st["queries"] = st["queries"].to(st["base"].dtype)
    return st


def _prepare_pq(case, seed):
    st = _graph_world(case, seed)
    base, m = st["base"], case["subspaces"]
    table = gi.train_pq(base, m, iters=4, sample=8192)
    codes = gi.pq_encode(base, table, m)
    st["table"] = table
    st["records"] = gs.SampleRecords.build(codes, *st["csr"])
    st["width"] = TOPK if case["inline"] else 100
    st["stats"] = torch.zeros(max(st["n_routes"], 1) * 8, dtype=torch.int32, device=DEV)
    st["sl"] = _route_rows(case, st["width"])
    return st


def _prepare_rabitq(case, seed):
    st = _graph_world(case, seed)
    base, P, nq = st["base"], _padded(case["dim"]), case["queries"]
    rot = _orthogonal(P, seed)[:case["dim"]].contiguous()
    centres = gi.train_kmeans(base, case["anchors"], iters=2, sample=16384, seed=9)
    codes, fac, aid, anchors = gi.rabitq_encode(base, rot, centres)
    rec = gs.RabitqRecords.build(codes, fac, aid, st["attr"], *st["csr"])
    A = int(anchors.shape[0])
    st["keep"] = (rot, codes, fac, aid, anchors, rec)
    st["rec"], st["rot"] = rec, rot
    st["rv"] = _lib.RabitqView(_lib.ptr(codes), _lib.ptr(fac), _lib.ptr(aid), _lib.ptr(anchors),
                               case["dim"], P, A, case["n"], *rec.view_fields())
    st["prep"] = (torch.empty(nq, P, device=DEV),
                  torch.empty(nq, P, dtype=torch.int8, device=DEV),
                  torch.empty(nq, device=DEV), torch.empty(nq, device=DEV),
                  torch.empty(nq, A, device=DEV))
    st["rq"] = _lib.RabitqQueries(*[_lib.ptr(t) for t in st["prep"]], nq)
    st["sl"] = _route_rows(case, case["width"])
    return st


def _one_bit(case, seed, nq):
    """One-bit codes of a base and prepared queries, in torch: the arrays a
    posting scan reads.  Codes are MSB-first in u32 words."""
    P, n, A = _padded(case["dim"]), case["n"], case["anchors"]
    base, queries = _vectors(case, seed, nq)
    rot = _orthogonal(P, seed)[:case["dim"]].contiguous()
    g = _gen(seed, 6)
    anchors = base[torch.randint(0, n, (A,), generator=g, device=DEV)] @ rot
    an = (anchors * anchors).sum(1)
    codes = torch.empty(n, P // 8, dtype=torch.uint8, device=DEV)
    fac = torch.empty(n, 3, device=DEV)
    aid = torch.empty(n, dtype=torch.int32, device=DEV)
    # bit 31 - d % 32 of little-endian word d / 32: byte 3 holds dims 0..7
    weight = 2 ** torch.arange(7, -1, -1, device=DEV, dtype=torch.int32)
    step = max(1, (1 << 27) // P)
    for s in range(0, n, step):
        x = base[s:s + step] @ rot
        a = torch.addmm(an[None, :], x, anchors.t(), alpha=-2.0).argmin(1)
        c = anchors[a]
        r = x - c
        bit = r > 0
        xu = torch.where(bit, 0.5, -0.5)
        l2, ipr, ipc = (r * r).sum(1), (r * xu).sum(1), (c * xu).sum(1)
        zero = ipr == 0
        ipr = torch.where(zero, torch.ones_like(ipr), ipr)
        fac[s:s + step, 0] = torch.where(zero, l2, l2 + 2.0 * l2 * (ipc / ipr))
        fac[s:s + step, 1] = torch.where(zero, torch.zeros_like(l2), -2.0 * l2 / ipr)
        fac[s:s + step, 2] = 0.0
        aid[s:s + step] = a.to(torch.int32)
        b = (bit.view(-1, P // 32, 4, 8).to(torch.int32) * weight).sum(-1).to(torch.uint8)
        codes[s:s + step] = b.flip(2).reshape(-1, P // 8)
    y = queries @ rot
    scale = (y.abs().amax(1) / 127.0).clamp_min(1e-20)
    q8 = (y / scale[:, None]).round().clamp_(-127, 127).to(torch.int8)
    k1 = -0.5 * y.sum(1)
    cd = ((y * y).sum(1)[:, None] + an[None, :] - 2.0 * y @ anchors.t()).clamp_min_(0.0)
    st = dict(ctx=_lib.Context(0), codes=codes, fac=fac, aid=aid, anchors=anchors, P=P,
              prep=(y.contiguous(), q8, scale, k1, cd.contiguous()))
    st["rv"] = _lib.RabitqView(_lib.ptr(codes), _lib.ptr(fac), _lib.ptr(aid), _lib.ptr(anchors),
                               case["dim"], P, A, n)
    st["rq"] = _lib.RabitqQueries(*[_lib.ptr(t) for t in st["prep"]], nq)
    return st


def _slices(case, rng):
    """Per route a narrow range of the attribute, about `rows` rows of n."""
    width = np.maximum(1.0, np.round(rng.uniform(0.5, 1.5, case["routes"]) * case["rows"] * ATTR /
                                     case["n"]))
    width = np.minimum(width, ATTR)
    lo = np.floor(rng.random(case["routes"]) * (ATTR - width + 1))
    return lo.astype(np.float32)[:, None], (lo + width).astype(np.float32)[:, None]


def _range_inputs(case, seed):
    rng = np.random.default_rng(seed * 1000 + 3)
    attr = rng.integers(0, ATTR, size=(case["n"], 1)).astype(np.float32)
    index = rp.RangePostingIndex.build(attr)
    lo, hi = _slices(case, rng)
    modes = np.full((case["routes"], 1), 3, np.uint8)
    off, size = rp.route_postings(index, rp.choose_slices(index, modes, lo, hi))
    return attr, index, modes, lo, hi, off, size


def _prepare_range_scan(case, seed):
    st = _one_bit(case, seed, case["routes"])
    attr, index, modes, lo, hi, off, size = _range_inputs(case, seed)
    ids = np.arange(case["routes"], dtype=np.uint32)
    st["segs"] = rp.DeviceSegments(rp.segment_plan(ids, off, size, 4096))
    st["post"] = index.device_postings()
    st["resident"] = index.resident_rows
    st["rows"] = rp.PostingRows(st["ctx"], st["rv"], st["post"], st["resident"])
    st["filter"] = [gs.u32(ids)] + [torch.from_numpy(a).to(DEV) for a in (modes, lo, hi, attr)]
    st["host"] = (off, size)
    return st


def _prepare_label_scan(case, seed):
    rng = np.random.default_rng(seed * 1000 + 3)
    st = _one_bit(case, seed, case["routes"])
    n, vocab = case["n"], case["labels"]
    cat = rng.choice(vocab, size=n, p=_zipf(vocab))
    tag = vocab + rng.integers(0, 20, size=n)
    attr = rng.integers(0, ATTR, size=(n, 1)).astype(np.float32)
    off, lab = _csr(np.stack([cat, tag], 1), vocab + 20)
    freq, post_off, post_ids = gi.postings_from_csr(off, lab, vocab + 20)
    li = gi.LabelIndex(vocab + 20, n, freq, np.zeros(vocab + 20, np.uint32),
                       np.zeros(vocab + 20, np.uint32), np.zeros(0, np.uint32),
                       np.zeros((0, 1), np.uint32), np.zeros(vocab + 20, np.uint32), post_off,
                       post_ids, off, lab, 1)
    # a conjunction of category, tag and a 1 to 10% range around some row
    row = rng.integers(0, n, size=case["routes"])
    wide = np.round(rng.uniform(0.01, 0.1, case["routes"]) * ATTR)
    lo = np.clip(attr[row, 0] - np.floor(rng.random(case["routes"]) * wide), 0, ATTR - 1)
    rows = sorted((int(cat[r]), int(q), int(tag[r]), float(lo[q]), float(lo[q] + wide[q]))
                  for q, r in enumerate(row))
    routes = gp._routeset([(q, c, [t], [(0, 3, a, b)]) for c, q, t, a, b in rows], li)
    st["dg"] = gs.DeviceGraph.upload(li)
    st["dr"] = gs.DeviceRoutes.upload(routes, attr)
    st["pv"] = st["dr"].predicate_view(st["dg"], 0.0, False)
    # the postings in posting order, cut in segments, shared where routes
    # re-read them
    group = routes.route_group.astype(np.int64)
    size = freq[group].astype(np.uint64)
    plan = rp.segment_plan(np.arange(routes.count), post_off[group].astype(np.uint64), size, 32768)
    total = int(post_off[vocab])
    st["post"], st["total"] = st["dg"].posting_ids, total
    st["rows"] = rp.PostingRows(st["ctx"], st["rv"], st["post"], total)
    st["cols"] = rp.PostingPredicateColumns(st["ctx"], st["pv"], st["post"], total)
    st["segs"] = rp.DeviceSegments(plan)
    used = int(freq[np.unique(group)].sum())
    st["share"] = None
    if int(size.sum()) >= 4 * used and st["P"] <= 1024:
        st["share"] = rp.DeviceShare(rp.share_plan(plan))
    st["host"] = (rows, off, lab, attr, post_off, post_ids)
    return st


def _prepare_exact_scan(case, seed):
    base, queries = _vectors(case, seed, case["routes"])
    attr, index, _, lo, hi, off, size = _range_inputs(case, seed)
    li = gi.LabelIndex(1, case["n"], np.array([case["n"]]), np.zeros(1, np.uint32),
                       np.zeros(1, np.uint32), np.zeros(0, np.uint32), np.zeros((0, 1), np.uint32),
                       np.zeros(1, np.uint32), np.array([0, case["n"]], np.uint64),
                       np.arange(case["n"], dtype=np.uint32),
                       np.arange(case["n"] + 1, dtype=np.uint32), np.zeros(case["n"], np.uint32), 1)
    rows = [(q, 0, [], [(0, 3, float(lo[q, 0]), float(hi[q, 0]))]) for q in range(case["routes"])]
    st = dict(ctx=_lib.Context(0), base=base, queries=queries.to(base.dtype),
              dg=gs.DeviceGraph.upload(li),
              dr=gs.DeviceRoutes.upload(gp._routeset(rows, li), attr), post=index.device_postings(),
              off=gs.u32(off.astype(np.uint32)), size=gs.u32(size.astype(np.uint32)),
              host=(off, size))
    st["pv"] = st["dr"].predicate_view(st["dg"], 0.0, False)
    return st


def _prepare_graph(case, seed):
    rng = np.random.default_rng(seed * 1000 + 3)
    base, _ = _vectors(case, seed, 1)
    off, lab, vocab, _ = _labels(dict(case, filter="pairs"), rng)
    return dict(be=gb.HipBuild(_lib.Context(0)), base=base, off=off, lab=lab, vocab=vocab)


def _prepare_codes(case, seed):
    base, _ = _vectors(case, seed, 1)
    st = dict(be=gb.HipBuild(_lib.Context(0)), base=base)
    if case["codec"] == "rabitq":
        st["rot"] = _orthogonal(_padded(case["dim"]), seed)[:case["dim"]].contiguous()
        g = _gen(seed, 6)
        pick = torch.randint(0, case["n"], (case["anchors"],), generator=g, device=DEV)
        st["centres"] = base[pick].float()
    return st


def prepare(case, seed):
    return dict(globals()["_prepare_" + case["kind"]](case, seed), case=dict(case))


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def _merge(st):
    return gs.merge_routes_gpu(st["ctx"], st["q_off"], st["q_routes"], st["ids"], st["dists"],
                               TOPK, st["case"]["queries"], TOPK)


def _rerank(st, width):
    ctx, base = st["ctx"], st["base"]
    ctx.check(ctx.lib.gofann_exact_rerank(
        ctx.handle, _lib.ptr(base), ELEM[st["case"]["elem"]], base.shape[1], base.shape[0],
        _lib.ptr(st["queries"]), _lib.ptr(st["dr"].route_query), _lib.ptr(st["sl"][0]), width,
        st["n_routes"], TOPK, _lib.ptr(st["ids"]), _lib.ptr(st["dists"])))


def _run_exact(st):
    ctx, base, case = st["ctx"], st["base"], st["case"]
    prm = _lib.ExactParams(case["beam"], 1, _lib.EARLY_STOP_ADAPTIVE, 0, TOPK, _lib.PLACE_AUTO)
    ctx.check(ctx.lib.gofann_exact_search(
        ctx.handle, _lib.ptr(base), ELEM[case["elem"]], base.shape[1], base.shape[0],
        _lib.ptr(st["queries"]), st["dg"].view(), _lib.ptr(st["label_size"]),
        st["dr"].predicate_view(st["dg"], 0.0, False), st["dr"].routes_view(), prm,
        _lib.ptr(st["ids"]), _lib.ptr(st["dists"]), None))
    return (st["ids"], st["dists"], *_merge(st))


def _run_pq(st):
    case, w = st["case"], st["width"]
    prm = gs.search_params(queue_limit=case["beam"], result_width=w, inline_exact=case["inline"])
    pqv = gs.pq_view(st["records"], st["table"], st["base"] if case["inline"] else None)
    gs.run_pq_routes(st["ctx"], pqv, st["queries"], st["dg"], st["dr"], prm,
                     out=(*st["sl"], st["stats"]), records=st["records"])
    if case["inline"]:
        st["ids"], st["dists"] = st["sl"]
    else:
        _rerank(st, w)
    return (st["sl"][0], st["sl"][1], *_merge(st))


def _run_rabitq(st):
    ctx, case, dr = st["ctx"], st["case"], st["dr"]
    ctx.check(ctx.lib.gofann_rabitq_prepare_queries(ctx.handle, st["rv"], _lib.ptr(st["queries"]),
                                                    case["queries"], _lib.ptr(st["rot"]),
                                                    st["rq"]))
    prm = gs.search_params(queue_limit=case["beam"], result_width=case["width"])
    ctx.check(ctx.lib.gofann_rabitq_search(
        ctx.handle, st["rv"], st["rq"], st["dg"].view(),
        dr.predicate_view(st["dg"], 0.15, True, records=st["rec"]), dr.routes_view(), prm,
        _lib.ptr(st["sl"][0]), _lib.ptr(st["sl"][1]), None))
    _rerank(st, case["width"])
    return (st["sl"][1], st["dists"], *_merge(st))


def _run_range_scan(st):
    rq, modes, lo, hi, attr = st["filter"]
    routes = _lib.Routes(_lib.ptr(rq), None, None, None, None, _lib.ptr(modes), _lib.ptr(lo),
                         _lib.ptr(hi), _lib.ptr(attr), 1, st["case"]["routes"], None)
    return rp.rabitq_range_scan(st["ctx"], st["rv"], st["rq"], _lib.PredicateView(), routes,
                                st["post"], st["resident"], st["segs"], st["case"]["width"],
                                rows=st["rows"])


def _run_label_scan(st):
    return rp.rabitq_posting_scan_segments(
        st["ctx"], st["rv"], st["rq"], st["pv"], st["dr"].route_query, st["post"], st["total"],
        st["segs"], st["case"]["width"], rows=st["rows"], cols=st["cols"], share=st["share"])


def _run_exact_scan(st):
    order = _lib.EXACT_ORDER_SERIAL if st["case"]["order"] == "serial" else _lib.EXACT_ORDER_WARP
    return gs.exact_posting(st["ctx"], st["base"], st["queries"], st["dr"].route_query, st["post"],
                            st["off"], st["size"], TOPK, order, st["pv"])


def _run_graph(st):
    case, be = st["case"], st["be"]
    centres = gi.train_kmeans(st["base"], case["centres"], iters=4, sample=32768, backend=be)
    li = gi.build_label_index(st["base"], st["off"], st["lab"], st["vocab"], centres,
                              case["degree"], threshold=100, backend=be)
    return (centres, *(torch.from_numpy(a.view(np.int32)) for a in
                       (li.graph, li.seed_local, li.row_to_sample)))


def _run_codes(st):
    case, be, x = st["case"], st["be"], st["base"]
    if case["codec"] == "pq":
        table = gi.train_pq(x, case["subspaces"], iters=6, sample=16384, backend=be)
        return table, gi.pq_encode(x, table, case["subspaces"], backend=be)
    codes, fac, aid, anchors = gi.rabitq_encode(x, st["rot"], st["centres"], backend=be)
    return codes, fac[:, :2].contiguous(), aid, anchors


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _route_count(case):
    # two routes for an AND of two tags; one per interval a range overlaps
    return case["queries"] * {"tags": 1.45, "interval": 1.6, "range": 1.0}[case["filter"]]


def work(case):
    kind, dim = case["kind"], case["dim"]
    if kind in ("exact", "pq", "rabitq"):
        R, r = case["degree"], _route_count(case)
        # a beam expands nodes in proportion to its width and scores the
        # neighbours of each that it has not seen (0.6 of them, measured);
        # a large batch reads every row and node of the index, once
        E, fresh = 0.75 * case["beam"] + 25.0, 0.6 * R
        row = dim * SIZE[case["elem"]]
        nodes = case["n"] * {"tags": 1.8, "interval": 2.0, "range": 1.0}[case["filter"]]
        graph = min(r * E, nodes) * (8 * R + 4)

        def once(count, size):
            return min(count, case["n"]) * size

        if kind == "exact":
            return dict(bytes=graph + once(r * E * fresh, row + 16) + r * (row + 8 * TOPK),
                        flops=r * E * fresh * 3 * dim)
        if kind == "pq":
            m = case["subspaces"]
            rank = E if case["inline"] else 100
            return dict(bytes=graph + once(r * E * fresh, m + 16) + once(r * rank, row) +
                        r * (row + 8 * TOPK), flops=r * (E * fresh * 3 * dim + rank * 3 * dim))
        P = _padded(dim)
        q, A, w = case["queries"], case["anchors"], case["width"]
        return dict(bytes=graph + once(r * E * fresh, P / 8 + 32) + once(r * w, row) +
                    4 * dim * P + 4 * A * P + q * (4 * dim + 5 * P + 4 * A) + r * 8 * w,
                    flops=r * (E * fresh * 2 * P + w * 3 * dim) + 2 * q * P * (dim + A))
    if kind == "range_scan":
        rows = case["routes"] * min(case["rows"], case["n"])
        P = _padded(dim)
        # the postings are shared by routes, so no row need be read twice
        return dict(bytes=min(rows, case["n"]) * (P / 8 + 20) +
                    case["routes"] * (P + 4 * case["anchors"] + 8 * case["width"]),
                    flops=rows * 2.0 * P)
    if kind == "label_scan":
        p = _zipf(case["labels"])
        rows = case["routes"] * case["n"] * float((p * p).sum())
        P = _padded(dim)
        return dict(bytes=case["n"] * (P / 8 + 40) +
                    case["routes"] * (P + 4 * case["anchors"] + 8 * case["width"]),
                    flops=rows * (0.003 * 2.0 * P + 4))
    if kind == "exact_scan":
        rows = case["routes"] * min(case["rows"], case["n"])
        row = dim * SIZE[case["elem"]]
        return dict(bytes=min(rows, case["n"]) * (row + 8) + case["routes"] * (row + 8 * TOPK),
                    flops=rows * 3.0 * dim)
    n, row = case["n"], dim * SIZE[case["elem"]]
    if kind == "graph":
        # rows (two tags each) against the rows of their bucket, every
        # row and the training sample against every centre
        per = 2.0 * n / case["labels"] / case["centres"]
        flops = 2.0 * n * per * 3 * dim + 2.0 * (n + 8 * 32768) * case["centres"] * dim
        return dict(bytes=n * row + 2.0 * n * (4 * case["degree"] + 8), flops=flops)
    if case["codec"] == "pq":
        return dict(bytes=n * (row + case["subspaces"]) + 16384 * row,
                    flops=(n + 6 * 16384) * 256 * 3.0 * dim)
    P = _padded(dim)
    return dict(bytes=n * (row + P / 8 + 16) + 4 * dim * P,
                flops=2.0 * n * P * (dim + case["anchors"]))


# ---------------------------------------------------------------------------
# Tolerances and 64-bit results
# ---------------------------------------------------------------------------
def tolerance(case):
    if case["kind"] == "rabitq":
        # the query rotation is a matrix product in 32 bits: another order
        # of its sums moves a few of a query's 8-bit components by one, and
        # with them estimates, beams and shortlists (queries moved by one
        # rounding: estimates 1e-5 apart, the same ids)
        return {"rel": 4e-5, "differ": 1e-3}
    if case["kind"] == "codes" and case["codec"] == "rabitq":
        # the rotation again: bits of components near zero, factors
        return {"rel": 1e-4, "differ": 1e-3}
    # every other path fixes the order of its sums, so results are the same
    # bit for bit
    return "exact"


def _top(dist, ids, k):
    """The k least (distance, id) pairs, ids distinct, padded."""
    order = np.lexsort((ids, dist))[:k]
    oi = np.full(k, -1, np.int32)
    od = np.full(k, np.finfo(np.float32).max, np.float64)
    oi[:len(order)], od[:len(order)] = ids[order], dist[order]
    return oi, od


def _bits(codes, P):
    """MSB-first code words as 0/1 float64 [rows][P]."""
    b = codes.view(-1, P // 32, 4).flip(2).unsqueeze(-1)
    sh = torch.arange(7, -1, -1, device=codes.device, dtype=torch.uint8)
    return ((b >> sh) & 1).reshape(-1, P).double()


def _estimates(st, q, ids):
    """One-bit distance estimates of rows `ids` for prepared query q."""
    _, q8, scale, k1, cd = st["prep"]
    ip = _bits(st["codes"][ids], st["P"]) @ q8[q].double()
    f = st["fac"][ids].double()
    g = cd[q].double()[st["aid"][ids].long()]
    return (f[:, 1] * (ip * scale[q].double() + k1[q].double()) + f[:, 0] + g).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "codes":
        if case["codec"] == "pq":
            return None  # k-means training: a fixed point of rounded means
        st = _prepare_codes(case, seed)
        x, rot = st["base"], st["rot"].double()
        anchors = st["centres"].double() @ rot
        an = (anchors * anchors).sum(1)
        fac, aid = [], []
        for s in range(0, case["n"], 1 << 16):
            xr = x[s:s + (1 << 16)].double() @ rot
            a = (an[None, :] - 2.0 * xr @ anchors.t()).argmin(1)
            c = anchors[a]
            r = xr - c
            xu = torch.where(r > 0, 0.5, -0.5).double()
            l2, ipr, ipc = (r * r).sum(1), (r * xu).sum(1), (c * xu).sum(1)
            ipr = torch.where(ipr == 0, torch.full_like(ipr, torch.inf), ipr)
            fac.append(torch.stack([l2 + 2.0 * l2 * (ipc / ipr), -2.0 * l2 / ipr], 1))
            aid.append(a.to(torch.int32))
        return None, torch.cat(fac), torch.cat(aid), anchors
    if kind == "exact_scan":
        st = _prepare_exact_scan(case, seed)
        off, size = (a.astype(np.int64) for a in st["host"])
        post = st["post"].long()
        oi, od = [], []
        for q in range(case["routes"]):
            ids = post[off[q]:off[q] + size[q]]
            d = st["base"][ids].double() - st["queries"][q].double()
            i, v = _top((d * d).sum(1).cpu().numpy(), ids.cpu().numpy(), TOPK)
            oi.append(i)
            od.append(v)
        return (torch.from_numpy(np.concatenate(oi)), torch.from_numpy(np.concatenate(od)),
                torch.from_numpy(size.astype(np.int32)))
    if kind == "range_scan":
        st = _prepare_range_scan(case, seed)
        off, size = (a.astype(np.int64) for a in st["host"])
        post = st["post"].long()
        rows = [post[o:o + s] for o, s in zip(off, size)]
        query = range(case["routes"])
        passes = size.astype(np.int32)
    elif kind == "label_scan":
        st = _prepare_label_scan(case, seed)
        spec, off, lab, attr, post_off, post_ids = st["host"]
        tag = torch.from_numpy(lab[off[:-1].astype(np.int64) + 1].astype(np.int64)).to(DEV)
        at = torch.from_numpy(attr[:, 0]).to(DEV)
        ids = torch.from_numpy(post_ids.astype(np.int64)).to(DEV)
        rows, query = [], []
        for c, q, t, a, b in spec:
            m = ids[int(post_off[c]):int(post_off[c + 1])]
            rows.append(m[(tag[m] == t) & (at[m] >= a) & (at[m] < b)])
            query.append(q)
        passes = np.array([len(r) for r in rows], np.int32)
    else:
        return None  # a beam's rows are those its own rounded distances led it to
    k = case["width"]
    tops = [_top(_estimates(st, q, r), r.cpu().numpy(), k) for q, r in zip(query, rows)]
    return (torch.from_numpy(np.stack([t[0] for t in tops])),
            torch.from_numpy(np.stack([t[1] for t in tops])), torch.from_numpy(passes))
