"""GPU parity of the fused filtered top-k against the closed-form oracle.

The oracle (orc.topk_bruteforce) computes exact fp64 squared L2 distances over
the passing ids and keeps the k smallest, ties broken by the smaller id.  The
GPU computes fp32 distances on MFMA tiles.  The bar: every returned distance
within 1e-4 relative of the fp64 distance of the returned id; distances
ascending; and the returned id set equal to the oracle's except for ids whose
distance ties the k-th distance within that tolerance.
"""
import numpy as np
import pytest

import orc
from helpers import mt_bernoulli

pytestmark = pytest.mark.gpu

RTOL = 1e-4


def _say(*a):
    print("CASE", *a, flush=True)


def _torch():
    import torch
    return torch


def _data(n_base, n_q, dim, seed):
    rng = np.random.default_rng(seed)
    base = rng.standard_normal((n_base, dim)).astype(np.float32)
    queries = rng.standard_normal((n_q, dim)).astype(np.float32)
    return base, queries


def _run(gpu, base, queries, k, filt):
    torch = _torch()
    db = torch.from_numpy(base).cuda()
    dq = torch.from_numpy(queries).cuda()
    dist = torch.empty((queries.shape[0], k), dtype=torch.float32, device="cuda")
    ids = torch.empty((queries.shape[0], k), dtype=torch.int64, device="cuda")
    gpu.topk_filtered(db, dq, k, filt, dist, ids)
    torch.cuda.synchronize()
    return dist.cpu().numpy(), ids.cpu().numpy()


def check_topk(base, queries, k, passing, got_d, got_i):
    want_d, want_i = orc.topk_bruteforce(base, queries, k, passing)
    n_pass = base.shape[0] if passing is None else int(np.count_nonzero(passing))
    valid = min(k, n_pass)
    for q in range(queries.shape[0]):
        gi, gd = got_i[q], got_d[q]
        assert np.all(gi[valid:] == -1) and np.all(np.isinf(gd[valid:])), f"query {q}: padding"
        gi, gd = gi[:valid], gd[:valid]
        assert np.all(gi >= 0) and np.all(gi < base.shape[0]), f"query {q}: id range"
        assert len(set(gi.tolist())) == valid, f"query {q}: duplicate ids"
        if passing is not None:
            assert np.all(passing[gi] != 0), f"query {q}: id outside the filter"
        exact = ((base[gi].astype(np.float64) - queries[q].astype(np.float64)) ** 2).sum(axis=1)
        assert np.allclose(gd, exact, rtol=RTOL, atol=0), f"query {q}: distance off by more than 1e-4 rel"
        assert np.all(np.diff(gd) >= 0), f"query {q}: not ascending"
        wi, wd = want_i[q][:valid], want_d[q][:valid]
        if valid == 0:
            continue
        kth = wd[-1]
        only_gpu = set(gi.tolist()) - set(wi.tolist())
        only_cpu = set(wi.tolist()) - set(gi.tolist())
        for i in only_gpu | only_cpu:
            di = float(((base[i].astype(np.float64) - queries[q].astype(np.float64)) ** 2).sum())
            assert abs(di - kth) <= RTOL * max(abs(kth), 1e-30), \
                f"query {q}: id {i} differs from the oracle and is not a tie at the k-th distance"


def _filter_from(gpu, kind, n_base, density, seed):
    """(device filter or None, passing mask as uint8) for the filter layouts under test."""
    if kind == "none":
        return None, None
    rng = np.random.default_rng(seed)
    ids = np.nonzero(rng.random(n_base) < density)[0].astype(np.uint32)
    mask = np.zeros(n_base, np.uint8)
    mask[ids] = 1
    if kind == "ids":  # all-bitmap, universe = n_base (negated above 50%)
        g = gpu.upload_from_ids(ids, n_base)
    elif kind == "keep":  # array / bitmap containers
        lt = orc.Lite.from_sorted_ids(ids)
        g = gpu.upload_containers(lt.containers(), n_base, False, lt.cardinality(), orc.PROMOTE_KEEP_DEFAULT)
    elif kind == "runs":
        run_ids = np.concatenate([np.arange(s, min(n_base, s + 700)) for s in range(0, n_base, 2000)])
        run_ids = run_ids.astype(np.uint32)
        mask = np.zeros(n_base, np.uint8)
        mask[run_ids] = 1
        lt = orc.Lite.from_sorted_ids(run_ids).run_optimize()
        g = gpu.upload_containers(lt.containers(), 0, False, 0, orc.PROMOTE_KEEP_DEFAULT)
    elif kind == "setop":  # a set-operation result: no key_index, max_key 0 (found by key search)
        other = np.nonzero(rng.random(n_base) < 0.6)[0].astype(np.uint32)
        ga = gpu.upload_from_ids(ids, n_base)
        gb = gpu.upload_from_ids(other, n_base)
        g = gpu.set_operation(ga, gb, gpu.AND)
        gpu.free(ga)
        gpu.free(gb)
        assert not g.key_index
        mask = np.zeros(n_base, np.uint8)
        mask[np.intersect1d(ids, other)] = 1
    elif kind == "beyond":  # filter ids past n_base are ignored
        extra = np.arange(n_base, n_base + 5000, dtype=np.uint32)
        g = gpu.upload_from_ids(np.concatenate([ids, extra]), n_base + 70000)
    else:
        raise ValueError(kind)
    return g, mask


CASES = [
    # (n_base, n_q, dim, k, filter kind, density, seed)
    (5000, 40, 128, 10, "none", 1.0, 1),
    (5000, 40, 128, 100, "none", 1.0, 2),
    (20000, 300, 128, 10, "ids", 0.3, 3),
    (20000, 64, 128, 100, "ids", 0.7, 4),  # negated filter
    (150000, 33, 128, 100, "keep", 0.01, 5),
    (150000, 33, 128, 10, "keep", 0.4, 6),
    (140000, 20, 128, 50, "runs", 0.0, 7),
    (30000, 16, 128, 10, "beyond", 0.2, 8),
    (3000, 10, 64, 256, "none", 1.0, 9),
    (4000, 12, 100, 30, "ids", 0.5, 10),
    (4000, 12, 17, 30, "none", 1.0, 11),
    (2500, 7, 32, 10, "keep", 0.002, 12),  # fewer passing ids than k
    (70000, 520, 128, 10, "none", 1.0, 13),  # three query blocks
    (16384, 40, 128, 100, "none", 1.0, 14),  # the small-set limit exactly
    (16385, 40, 128, 100, "none", 1.0, 15),  # one row past it
    (3000, 9, 64, 10, "keep", 0.0, 16),  # no passing row: every slot is (+inf, -1)
    (60000, 20, 64, 10, "setop", 0.3, 17),
    (5000, 20, 17, 10, "keep", 0.3, 18),  # a filter with scalar row loads (dim % 4 != 0)
    (50000, 20, 72, 10, "ids", 0.4, 19),  # a filter, dim 72 of the 128-wide tiles
    (41000, 30, 128, 40, "setop", 0.5, 20),  # a filtered list path with a partial last tile in every chunk
]


SMALL_LIMITS = {"lists": 0, "small_16384": 16384, "small_default": 1 << 18}


@pytest.fixture(params=list(SMALL_LIMITS))
def path(request, gpu):
    """Runs a test with the limit at 0 (every case on the per-chunk sorted lists),
    at 16384 passing rows (both sides of it in the cases below), and with the
    default limit (estimates kept, or candidates under a bound)."""
    prev = gpu.topk_set_small_limit(SMALL_LIMITS[request.param])
    yield request.param
    gpu.topk_set_small_limit(prev)


@pytest.mark.parametrize("n_base,n_q,dim,k,kind,density,seed", CASES)
def test_topk_parity(gpu, path, n_base, n_q, dim, k, kind, density, seed):
    _say("topk", path, n_base, n_q, dim, k, kind, density, seed)
    base, queries = _data(n_base, n_q, dim, seed)
    filt, mask = _filter_from(gpu, kind, n_base, density, seed)
    got_d, got_i = _run(gpu, base, queries, k, filt)
    check_topk(base, queries, k, mask, got_d, got_i)
    if filt is not None:
        gpu.free(filt)


def test_topk_ties_break_by_id(gpu, path):
    """Duplicate base vectors tie exactly; the smaller id comes first."""
    _say("topk ties")
    rng = np.random.default_rng(21)
    uniq = rng.standard_normal((50, 128)).astype(np.float32)
    base = np.repeat(uniq, 40, axis=0)  # 2000 rows, each vector 40 times
    perm = rng.permutation(base.shape[0])
    base = np.ascontiguousarray(base[perm])
    queries = np.ascontiguousarray(uniq[:5] + 0.01 * rng.standard_normal((5, 128)).astype(np.float32))
    got_d, got_i = _run(gpu, base, queries, 60, None)
    check_topk(base, queries, 60, None, got_d, got_i)
    for q in range(5):
        for a in range(59):
            if got_d[q, a] == got_d[q, a + 1]:
                assert got_i[q, a] < got_i[q, a + 1]


def test_topk_multi_and_filter(gpu, path):
    """The workload's shape: filter = multi_and of three predicates."""
    _say("topk multi_and filter")
    n_base = 200000
    preds = [mt_bernoulli(60 + i, 0.5, n_base) for i in range(3)]
    gs = [gpu.upload_from_ids(p, n_base) for p in preds]
    f = gpu.multi_and(gs)
    mask = np.ones(n_base, np.uint8)
    for p in preds:
        m = np.zeros(n_base, np.uint8)
        m[p] = 1
        mask &= m
    base, queries = _data(n_base, 24, 128, 61)
    got_d, got_i = _run(gpu, base, queries, 10, f)
    check_topk(base, queries, 10, mask, got_d, got_i)
    for g in gs + [f]:
        gpu.free(g)


@pytest.mark.parametrize("rows", [16384, 16385, 24003, 40960, 40961])
@pytest.mark.parametrize("filtered", [False, True])
def test_topk_kept_estimates(gpu, rows, filtered):
    """Every estimate is kept up to 40960 rows here (64 dimensions or fewer, at most
    256 queries); past it the sample and candidate lists answer."""
    _say("topk kept estimates", rows, filtered)
    n_base = rows + 9000 if filtered else rows
    mask = np.ones(n_base, np.uint8)
    if filtered:
        mask[np.random.default_rng(rows).choice(n_base, 9000, replace=False)] = 0
    base, queries = _data(n_base, 70, 48, rows)
    g = gpu.upload_from_ids(np.flatnonzero(mask).astype(np.uint32), n_base) if filtered else None
    for n_q, k in ((5, 3), (70, 100)):
        got_d, got_i = _run(gpu, base, queries[:n_q], k, g)
        check_topk(base, queries[:n_q], k, mask, got_d, got_i)
    if filtered:
        gpu.free(g)


@pytest.mark.parametrize("n_q,k", [(2, 10), (9, 256), (64, 33), (70, 10)])
@pytest.mark.parametrize("n_base", [100000, 2200000])
def test_topk_two_far_modes(gpu, n_base, n_q, k):
    """Half of the rows and every second query 4000 away from the others: one
    point is a centre for one half only, and every near row is a candidate of the
    other half's queries, whose selection is split over several workgroups (up to 64
    queries; the larger set's lists cannot hold every row)."""
    _say("topk two modes", n_base, n_q, k)
    base, queries = _data(n_base, n_q, 16, 59)
    base[1::2] += 1000
    queries[1::2] += 1000
    got_d, got_i = _run(gpu, base, queries, k, None)
    pick = np.arange(0, n_q, 1 + n_q // 6)
    check_topk(base, queries[pick], k, None, got_d[pick], got_i[pick])


@pytest.mark.parametrize("n_base,n_q", [(9000, 5), (24576, 70), (60000, 5), (60000, 300), (300000, 9)])
@pytest.mark.parametrize("shift", [0.0, 300.0])
def test_topk_equal_rows(gpu, shift, n_base, n_q):
    """Every row the same: all estimates fall into one bin, more rows than a batch
    holds lie at the edge, and the smallest ids are the answer."""
    _say("topk equal rows", shift, n_base, n_q)
    row, queries = _data(1, n_q, 40, 61)
    base = np.repeat(row + np.float32(shift), n_base, axis=0)
    got_d, got_i = _run(gpu, base, queries + np.float32(shift), 20, None)
    assert np.array_equal(got_i, np.broadcast_to(np.arange(20), (n_q, 20)))
    assert np.all(got_d == got_d[:, :1])
    exact = ((base[0].astype(np.float64) - (queries + np.float32(shift)).astype(np.float64)) ** 2).sum(axis=1)
    assert np.allclose(got_d[:, 0], exact, rtol=RTOL, atol=0)


def test_topk_four_far_modes(gpu):
    """Rows and queries in four modes, none near the block's centre: every query goes
    from the sample to the list path, but for a block whose queries share one mode."""
    _say("topk four modes")
    n_base, n_q = 600000, 300
    base, queries = _data(n_base, n_q, 16, 60)
    for m in range(4):
        base[m::4, 4 * m:4 * m + 4] += 1000
        queries[m:256:4, 4 * m:4 * m + 4] += 1000
    queries[256:, :4] += 1000
    got_d, got_i = _run(gpu, base, queries, 10, None)
    pick = np.arange(0, n_q, 23)
    check_topk(base, queries[pick], 10, None, got_d[pick], got_i[pick])


@pytest.mark.parametrize("n_q,most", [(1, 80), (20, 160)])
def test_topk_scratch_of_few_queries(gpu, n_q, most):
    """The candidate lists are sized for the queries there are and the candidates to
    expect: 2 MB a query, beside 4 MB of estimates (512 MB when 64 queries' lists of
    2048 each were taken for any number)."""
    _say("topk scratch", n_q)
    torch = _torch()
    base = torch.randn(3_000_000, 32, device="cuda")
    q = torch.randn(n_q, 32, device="cuda")
    d = torch.empty(n_q, 10, device="cuda")
    i = torch.empty(n_q, 10, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    gpu.load().cr_mempool_trim(-1, 0)
    before = torch.cuda.mem_get_info()[0]
    gpu.topk_filtered(base, q, 10, None, d, i)
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] < most << 20


@pytest.mark.parametrize("n_q,dim,rows", [(4, 128, 65536), (4, 128, 65537), (256, 65, 65536), (257, 65, 40960),
                                          (257, 64, 40961), (512, 32, 24577), (513, 32, 24576), (513, 96, 24577)])
def test_topk_kept_limits(gpu, n_q, dim, rows):
    """Both sides of the limits of the kept rows: 65536 (up to 256 queries of more
    than 64 dimensions), 40960 (up to 512 queries), 24576."""
    _say("topk kept limits", n_q, dim, rows)
    base, queries = _data(rows, n_q, dim, rows + n_q)
    got_d, got_i = _run(gpu, base, queries, 33, None)
    pick = np.arange(0, n_q, 1 + n_q // 20)
    check_topk(base, queries[pick], 33, None, got_d[pick], got_i[pick])


def test_topk_understated_cardinality(gpu):
    """The host leaves the list path out when a filter's recorded cardinality
    fits the small-set limit.  A caller-built struct whose total_cardinality
    understates its set (the library's own results record the exact count) then
    reaches tk_select with more rows than the limit, which takes every passing
    row as a candidate: the answer is still exact."""
    _say("topk understated cardinality")
    prev = gpu.topk_set_small_limit(16384)
    try:
        n_base = 60000
        ids = mt_bernoulli(71, 0.5, n_base)  # ~30000 passing rows, past the limit
        g = gpu.upload_from_ids(ids, n_base)
        true_card = g.total_cardinality
        assert true_card > 16384
        g.total_cardinality = 100
        mask = np.zeros(n_base, np.uint8)
        mask[ids] = 1
        base, queries = _data(n_base, 12, 64, 72)
        got_d, got_i = _run(gpu, base, queries, 20, g)
        check_topk(base, queries, 20, mask, got_d, got_i)
        g.total_cardinality = true_card
        gpu.free(g)
    finally:
        gpu.topk_set_small_limit(prev)


def test_topk_rejects_unsupported(gpu):
    _say("topk unsupported")
    torch = _torch()
    base = torch.zeros((10, 200), device="cuda")
    q = torch.zeros((2, 200), device="cuda")
    d = torch.empty((2, 5), device="cuda")
    i = torch.empty((2, 5), dtype=torch.int64, device="cuda")
    with pytest.raises(gpu.CrError):
        gpu.topk_filtered(base, q, 5, None, d, i)


@pytest.fixture
def keep16384(gpu):
    """At most 16384 rows keep their estimates, whatever the number of queries:
    larger sets go through the sample and the candidate kernel."""
    prev = gpu.topk_set_small_limit(16384)
    yield
    gpu.topk_set_small_limit(prev)


# The estimate path past its kept rows (16384 here): each padded dimension count
# and its edges, both workgroup shapes (up to 64 queries, and 256 a workgroup
# with partial groups), one and two candidate stages (k rows > 1024 x 16384, or
# times the queries > 2^17 x 16384) of either shape, with a filter and without, a
# partial last tile, and exactly one row more than is kept.
GATED = [
    # (n_base, n_q, dim, k, filter kind, density, seed)
    (16385, 1, 32, 1, "none", 1.0, 31),
    (16385, 257, 31, 5, "none", 1.0, 32),
    (40001, 65, 64, 3, "none", 1.0, 33),
    (40063, 64, 33, 7, "none", 1.0, 34),
    (50000, 100, 96, 10, "ids", 0.9, 35),
    (33000, 30, 65, 10, "keep", 0.8, 36),
    (20000, 20, 97, 256, "none", 1.0, 37),
    (180000, 70, 96, 100, "none", 1.0, 38),  # two stages
    (300000, 9, 20, 200, "ids", 0.6, 39),  # two stages, a negated filter, few queries
    (600000, 3, 17, 256, "none", 1.0, 40),
    (200000, 300, 64, 60, "ids", 0.5, 41),  # two stages, a filter, two blocks of 256 queries
    (220000, 130, 128, 150, "keep", 0.4, 42),  # the same with key-searched ids, a partial query group
]


@pytest.mark.parametrize("n_base,n_q,dim,k,kind,density,seed", GATED)
def test_topk_gated(gpu, keep16384, n_base, n_q, dim, k, kind, density, seed):
    _say("topk gated", n_base, n_q, dim, k, kind, density, seed)
    base, queries = _data(n_base, n_q, dim, seed)
    filt, mask = _filter_from(gpu, kind, n_base, density, seed)
    got_d, got_i = _run(gpu, base, queries, k, filt)
    check_topk(base, queries, k, mask, got_d, got_i)
    if filt is not None:
        gpu.free(filt)


@pytest.mark.parametrize("n_q", [20, 90])
@pytest.mark.parametrize("scale", [1e-8, 1e-3, 1e3, 1e8])
def test_topk_gated_scales(gpu, keep16384, scale, n_q):
    """The split's scale follows each vector's norm: rows of very different
    norms in one set, at magnitudes far outside the range of 16-bit floats."""
    _say("topk scales", scale, n_q)
    base, queries = _data(30000, n_q, 128, 51)
    base *= np.float32(scale) * np.exp2(np.arange(30000) % 23 - 11).astype(np.float32)[:, None]
    queries *= np.float32(scale)
    got_d, got_i = _run(gpu, base, queries, 20, None)
    check_topk(base, queries, 20, None, got_d, got_i)


@pytest.mark.parametrize("n_q", [8, 80])
@pytest.mark.parametrize("n_base", [3000, 30000])
def test_topk_unusual_rows(gpu, keep16384, n_base, n_q):
    """Rows and queries that the estimates leave out (zero, or of a norm that
    overflows or underflows) and rows with infinities or NaN: the finite
    distances are answered exactly, infinite ones come last, NaN never."""
    _say("topk unusual", n_base, n_q)
    base, queries = _data(n_base, n_q, 64, 53)
    base[5] = 0
    base[7] = queries[1]
    base[11] *= 1e-15
    base[13, 3] = np.inf
    base[17, 4] = -np.inf
    base[19, 5] = np.nan
    base[23] = 1e25
    queries[2] = 0
    queries[3] *= 1e-15
    got_d, got_i = _run(gpu, base, queries, 10, None)
    bad = np.isin(np.arange(n_base), [13, 17, 19, 23])
    mask = (~bad).astype(np.uint8)
    clean = base.copy()
    clean[bad] = 0
    check_topk(clean, queries, 10, mask, got_d, got_i)
    # fewer finite rows than k: the infinite distances fill up, the NaN row is left out
    few = np.array([5, 7, 13, 17, 19, 23])
    sub = np.ascontiguousarray(base[few])
    got_d, got_i = _run(gpu, sub, queries, 8, None)
    for q in range(n_q):
        assert set(got_i[q, :2].tolist()) == {0, 1} and np.all(np.isfinite(got_d[q, :2]))
        assert got_i[q, 2:5].tolist() == [2, 3, 5] and np.all(np.isinf(got_d[q, 2:5]))
        assert np.all(got_i[q, 5:] == -1) and np.all(np.isinf(got_d[q, 5:]))


@pytest.mark.parametrize("n_q", [9, 75])
@pytest.mark.parametrize("n_base,k", [(9000, 10), (30000, 10), (120000, 200)])
@pytest.mark.parametrize("far", [1e3, 1e6])
def test_topk_far_rows(gpu, keep16384, n_base, k, far, n_q):
    """A few rows at 10^6 and 10^12 times the others' distance, sampled ones among
    them: the histogram of the estimates holds nearly every row in its first bin
    and is taken again over that."""
    _say("topk far rows", n_base, k, far, n_q)
    base, queries = _data(n_base, n_q, 64, 57)
    base[::97] *= np.float32(far)
    got_d, got_i = _run(gpu, base, queries, k, None)
    pick = np.arange(0, n_q, 5)
    check_topk(base, queries[pick], k, None, got_d[pick], got_i[pick])


# (n_base, n_q, dim, k, filter kind, density): kept estimates, candidates in one
# stage and in two, with row loads of one float and of four, whole and partial
# blocks of either workgroup shape
OFF_CENTRE = [
    (9000, 5, 128, 10, "none", 1.0),
    (9000, 70, 33, 30, "ids", 0.6),
    (30000, 60, 100, 10, "none", 1.0),
    (40000, 300, 64, 10, "keep", 0.7),
    (200000, 1, 96, 100, "none", 1.0),
    (200000, 70, 31, 100, "ids", 0.8),
]


@pytest.mark.parametrize("n_base,n_q,dim,k,kind,density", OFF_CENTRE)
@pytest.mark.parametrize("shift", [20.0, 300.0])
def test_topk_off_centre(gpu, keep16384, shift, n_base, n_q, dim, k, kind, density):
    """Vectors far from the origin, where the estimates' margin is large beside the
    distances (300: beyond every distance in the set)."""
    _say("topk off centre", shift, n_base, n_q, dim, k, kind, density)
    base, queries = _data(n_base, n_q, dim, 58)
    move = np.float32(shift) * np.where(np.arange(dim) % 3 == 0, -1, 1).astype(np.float32)
    base += move
    queries += move
    filt, mask = _filter_from(gpu, kind, n_base, density, 58)
    got_d, got_i = _run(gpu, base, queries, k, filt)
    pick = np.arange(0, n_q, 7)
    check_topk(base, queries[pick], k, mask, got_d[pick], got_i[pick])
    if filt is not None:
        gpu.free(filt)


def test_topk_candidates_overflow(gpu):
    """Every sampled row is far from the queries and every other row near, so the
    sample bounds nothing and the candidate lists (bounded at this size)
    overflow: the list path answers."""
    _say("topk overflow")
    n, n_q = 200000, 1024
    base, queries = _data(n, n_q, 32, 55)
    base *= np.float32(0.1)
    queries *= np.float32(0.1)
    sampled = (np.arange(16384, dtype=np.uint64) * np.uint64(n)) >> np.uint64(14)
    base[sampled] += 50
    got_d, got_i = _run(gpu, base, queries, 10, None)
    pick = np.arange(0, n_q, 37)
    check_topk(base, queries[pick], 10, None, got_d[pick], got_i[pick])


def test_topk_some_queries_overflow(gpu):
    """One block of 256 queries where every third one's candidate lists overflow:
    those are near the rows that the sample leaves out, the others near the
    sampled ones.  The list path answers the former and leaves the latter."""
    _say("topk some overflow")
    n, n_q = 200000, 1024
    base, queries = _data(n, n_q, 32, 56)
    base *= np.float32(0.1)
    queries *= np.float32(0.1)
    sampled = (np.arange(16384, dtype=np.uint64) * np.uint64(n)) >> np.uint64(14)
    base[sampled] += 50
    queries[np.arange(n_q) % 3 != 0] += 50
    got_d, got_i = _run(gpu, base, queries, 10, None)
    pick = np.arange(0, n_q, 35)
    check_topk(base, queries[pick], 10, None, got_d[pick], got_i[pick])


@pytest.mark.parametrize("n_q", [1, 70])
def test_topk_second_bound_rounding(gpu, n_q):
    """The sampled rows bound the k-th distance by 1, the first tiles by less than
    1e-6 of that: the candidates of the first tiles are rounded at the size of
    the first bound, and nearer rows of the other tiles must still be answered."""
    _say("topk second bound", n_q)
    n, k = 100000, 256  # k n / 16384 > 1024: two stages
    row = np.arange(n)
    sampled = np.zeros(n, bool)
    sampled[(np.arange(16384, dtype=np.uint64) * np.uint64(n)) >> np.uint64(14)] = True
    first = row // 64 % 16 == 0  # the tiles that give the second bound
    d = np.full(n, 2.0)
    d[sampled & ~first] = 1.0
    d[np.flatnonzero(first & ~sampled)[:300]] = 8e-7
    nearest = np.flatnonzero(~first & ~sampled)[:50]
    d[nearest] = 5e-7
    base = np.zeros((n, 32), np.float32)
    base[:, 0] = np.sqrt(d)
    queries = np.zeros((n_q, 32), np.float32)
    got_d, got_i = _run(gpu, base, queries, k, None)
    check_topk(base, queries, k, None, got_d, got_i)
    assert np.array_equal(np.sort(got_i[:, :50], axis=1), np.broadcast_to(nearest, (n_q, 50)))
