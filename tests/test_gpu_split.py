"""Float32 batches on the two-piece fp16 route against the CPU restatement.

Large float32 batches multiply their rows as two binary16 pieces; the rows'
values decide on the device between the hi pieces alone, both pieces, and
the float32 kernels.  Every kind of values here must give what the float32
route gives: integers bit for bit (their sums are exact either way), real
values to float32 accuracy.

The tolerance on real values is one of each sum's own terms, sum |q_i b_i| (not
of the rows' lengths, which say nothing of a query that is zero where its rows
are large).  In units of 2^-24 of it: the pieces hold each value to 2 (both
sides: 4), the lo x lo products that may be left out are at most 4, a small
value's loss at most 1 (inner products; L2: 2 of |q| |b|), and the float32 sums,
on either unit, take at most one rounding a term: d + 9 in all.  L2 takes that
twice and adds its norms' and last sums' roundings, d + 4 of |q|^2 + |b|^2 at
most; cosine rounds each unit value, d / 8 + 6 a side.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N, NQ = 66_001, 4_003  # n nq max(d, 32) past the route's least work, ragged tiles and blocks
SAMPLE = 40            # queries checked: the first, the last and some between


def size_of(d):
    """Fewer rows and queries for long rows (the same matrix work)."""
    return (N, NQ) if d <= 256 else (30_011, 2_003)


def rows_of(kind, n, d, r):
    if kind == "bytes":        # 8-bit integers: the hi pieces alone
        return r.integers(0, 256, (n, d)).astype(np.float32)
    if kind == "halves":       # binary16 values, both signs
        return r.standard_normal((n, d)).astype(np.float16).astype(np.float32)
    if kind == "wide ints":    # 12-bit integers with lo pieces on both sides: lo x lo counts
        x = np.zeros((n, d), np.float32)
        x[np.arange(n), r.integers(0, min(d, 4), n)] = r.integers(2049, 2800, n)
        return x
    x = r.standard_normal((n, d)).astype(np.float32)
    if kind == "outlier":      # past binary16's range in the sample's scale: the float32 kernels
        x[n // 2, d // 2] = 3.0e6
    if kind == "tiny row":     # below the pieces' precision: the float32 kernels
        x[n // 3] *= np.float32(1e-9)
    if kind == "small":        # a scale far from 1
        x *= np.float32(2.0 ** -40)
    return x


def sample(nq, count=SAMPLE):
    edges = np.array([0, 1, 31, 32, 63, 64, 127, 128, nq - 1, nq - 2])
    return np.unique(np.concatenate([edges[edges < nq],
                                     np.linspace(0, nq - 1, count).astype(int)]))


def check(engine, oracle, base, q, k, metric, exact, count=SAMPLE, **filt):
    if filt:
        ids, dist = engine.brute_force_knn_filtered(base, q, k, metric, **filt)
    else:
        ids, dist = engine.brute_force_knn(base, q, k, metric)
    pick = sample(len(q), count)
    if base.dtype == np.float16:
        base, q = oracle.f16_to_f32(base), oracle.f16_to_f32(q)
    if filt:
        oi, od = oracle.knn_filtered(base, q[pick], k, metric, **filt)
    else:
        oi, od = oracle.knn(base, q[pick], k, metric)
    if exact:
        assert np.array_equal(ids[pick], oi)
        assert np.array_equal(dist[pick], od)
        return
    q64 = q[pick].astype(np.float64)
    bn = np.sqrt(np.einsum("ij,ij->i", base, base, dtype=np.float64))
    qn = np.linalg.norm(q64, axis=1)

    def products(f):
        return np.concatenate([f(base[i:i + 20_000].astype(np.float64)) @ f(q64).T
                               for i in range(0, len(base), 20_000)])

    dots, terms = products(lambda x: x), products(np.abs)
    d, u = base.shape[1], 2.0 ** -24
    for i in range(len(pick)):
        got, g = ids[pick][i], dist[pick][i].astype(np.float64)
        s, err = dots[:, i], (d + 9) * u * terms[:, i]
        if metric == "l2":
            s = bn * bn + qn[i] * qn[i] - 2 * s
            err = 2 * err + (d + 4) * u * (qn[i] ** 2 + bn * bn) + 2 * u * qn[i] * bn
        elif metric == "cosine":
            mag = np.maximum(qn[i] * bn, 1e-300)
            s, err = s / mag, (err + (d / 4 + 12) * u * terms[:, i]) / mag
        if "bitset" in filt:
            s = np.where(filt["bitset"], s, np.inf if metric == "l2" else -np.inf)
        assert len(set(got.tolist())) == k
        assert (np.abs(g - s[got]) <= err[got]).all(), (np.abs(g - s[got]) / err[got]).max()
        # no row left out is better than one kept by more than their two errors
        order = s if metric == "l2" else -s
        left = np.ones(len(s), bool)
        left[got] = False
        assert (order + err)[left].min() >= (order - err)[got].max()


@pytest.mark.parametrize("kind,metric,d,k,exact", [
    ("bytes", "l2", 128, 10, True),
    ("bytes", "l2", 99, 33, True),
    ("bytes", "inner_product", 64, 4, True),
    ("halves", "inner_product", 100, 10, False),
    ("wide ints", "l2", 128, 10, True),
    ("wide ints", "l2", 20, 8, True),
    ("float", "l2", 128, 10, False),
    ("float", "l2", 33, 1, False),
    ("float", "inner_product", 65, 16, False),
    ("float", "cosine", 96, 10, False),
    ("float", "cosine", 27, 40, False),
    ("float", "l2", 128, 100, False),
    ("small", "l2", 120, 10, False),
    ("outlier", "l2", 128, 10, False),
    ("outlier", "cosine", 128, 20, False),
    ("tiny row", "inner_product", 99, 10, False),
    ("tiny row", "l2", 36, 40, False),
    # the tile kernel: rows too long to hold a query's pieces in registers
    ("bytes", "l2", 130, 10, True),
    ("bytes", "inner_product", 200, 16, True),
    ("wide ints", "l2", 137, 10, True),
    ("wide ints", "l2", 300, 33, True),
    ("float", "l2", 129, 10, False),
    ("float", "inner_product", 256, 3, False),
    ("float", "cosine", 255, 40, False),
    ("float", "l2", 257, 40, False),
    ("float", "cosine", 384, 10, False),
    ("float", "cosine", 301, 40, False),
    ("float", "l2", 768, 16, False),
    ("outlier", "l2", 144, 10, False),
    ("outlier", "l2", 320, 16, False),
    ("outlier", "cosine", 384, 10, False),
    ("outlier", "cosine", 299, 10, False),
    ("outlier", "cosine", 299, 40, False),
    ("tiny row", "inner_product", 290, 40, False),
])
def test_every_kind_of_values(engine, oracle, kind, metric, d, k, exact):
    r = np.random.default_rng(d + k)
    n, nq = size_of(d)
    base, q = rows_of(kind, n, d, r), rows_of(kind, nq, d, r)
    check(engine, oracle, base, q, k, metric, exact)


@pytest.mark.parametrize("metric", ["inner_product", "cosine", "l2"])
@pytest.mark.parametrize("kind,d,scale", [
    ("columns", 128, 1e-6), ("columns", 128, 1e-10), ("columns", 40, 1e-8), ("columns", 768, 1e-8),
    ("rows", 128, 1e-6), ("rows", 300, 1e-8), ("rows", 64, 1e-3),
])
def test_small_values_decide(engine, oracle, metric, kind, d, scale):
    """Scores that rest on values far below the rest of the data: columns of a
    small scale under queries that are zero elsewhere, and sparse rows of small
    values; neither has many values that the pieces lose bits of."""
    r = np.random.default_rng(d)
    n, nq = size_of(d)
    base, q = rows_of("float", n, d, r), rows_of("float", nq, d, r)
    some = r.choice(d, d // 16, replace=False)
    if kind == "columns":
        base[:, some] *= np.float32(scale)
        keep = np.zeros(d, np.float32)
        keep[some] = 1
        q[::2] *= keep
    else:
        small = np.zeros((n // 8, d), np.float32)
        small[:, some] = base[:n // 8, some] * np.float32(scale)
        base[:n // 8] = small
        check(engine, oracle, base, q, 10, metric, False, bitset=np.arange(n) < n // 8)
    check(engine, oracle, base, q, 10, metric, False)


@pytest.mark.parametrize("d", [128, 48, 131, 300])
def test_integers_beside_long_ones(engine, oracle, d):
    """Sums of 12-bit integers are exact, also where other rows and other
    queries hold integers of 21 bits (and their own sums are not)."""
    r = np.random.default_rng(d)
    n, nq = size_of(d)
    base, q = rows_of("wide ints", n, d, r), rows_of("wide ints", nq, d, r)
    base[::8] *= 1001
    q[np.setdiff1d(np.arange(0, nq, 8), sample(nq))] *= 1001
    check(engine, oracle, base, q, 10, "l2", True)


@pytest.mark.parametrize("d", [128, 300])
def test_integers_of_24_bits(engine, oracle, d):
    """Inner products with unit vectors are the rows' own 24-bit integers."""
    r = np.random.default_rng(d)
    n, nq = size_of(d)
    base = r.integers(-(1 << 24) + 1, 1 << 24, (n, d)).astype(np.float32)
    q = np.zeros((nq, d), np.float32)
    q[np.arange(nq), r.integers(0, d, nq)] = 1
    check(engine, oracle, base, q, 10, "inner_product", True)


@pytest.mark.parametrize("kind,metric,d", [
    ("bytes", "cosine", 320),
    ("float", "l2", 16), ("float", "l2", 24), ("float", "l2", 40), ("float", "l2", 128),
    ("positive", "l2", 200), ("float", "l2", 768), ("float", "inner_product", 9),
    ("float", "inner_product", 33), ("positive", "inner_product", 300), ("float", "cosine", 96),
    ("float", "cosine", 384),
    # few terms that count, in long rows too; values whose products have few bits
    ("half zeros", "l2", 40), ("half zeros", "l2", 128), ("half zeros", "l2", 300),
    ("sparse", "l2", 96), ("sparse", "l2", 160), ("log-normal", "l2", 40), ("log-normal", "l2", 64),
    ("log-normal", "inner_product", 16), ("log-normal", "inner_product", 36),
    ("log-normal", "inner_product", 56), ("counts", "cosine", 36),
    ("sixty-fourths", "cosine", 320), ("bfloat16", "cosine", 512),
])
def test_errors_no_larger_than_the_float32_kernels(engine, kind, metric, d):
    """Errors against 64 bits of a batch and of its first 128 queries alone,
    which the float32 kernels take.  128 x 16 distances: their rms is known to
    1 / sqrt(2 x 2,048), 1.6%, so 6% is past chance."""
    r = np.random.default_rng(d)
    n, nq = size_of(d)
    make = {"positive": lambda *s: r.random(s, np.float32),
            "bytes": lambda *s: r.integers(0, 256, s).astype(np.float32),
            "half zeros": lambda *s: np.maximum(r.standard_normal(s, np.float32), 0),
            "sparse": lambda *s: np.abs(r.standard_normal(s, np.float32)) * (r.random(s) < 0.05),
            "log-normal": lambda *s: np.exp(r.standard_normal(s, np.float32)),
            "counts": lambda *s: r.poisson(0.5, s).astype(np.float32),
            "sixty-fourths": lambda *s: np.round(r.standard_normal(s, np.float32) * 64) / 64,
            "bfloat16": lambda *s: (r.standard_normal(s, np.float32).view(np.uint32)
                                    & np.uint32(0xffff0000)).view(np.float32),
            "float": lambda *s: r.standard_normal(s, np.float32)}[kind]
    base, q = make(n, d), make(nq, d)

    def rms(batch):
        ids, dist = engine.brute_force_knn(base, q[:batch], 16, metric)
        b, x = base[ids[:128]].astype(np.float64), q[:128, None].astype(np.float64)
        if metric == "l2":
            want = ((b - x) ** 2).sum(2)
        else:
            want = (b * x).sum(2)
            if metric == "cosine":
                want /= np.maximum(np.linalg.norm(b, axis=2) * np.linalg.norm(x, axis=2), 1e-30)
        return np.sqrt(((dist[:128] - want) ** 2).mean())

    assert rms(nq) <= 1.06 * rms(128)


@pytest.mark.parametrize("metric,d,eb,eq", [
    ("inner_product", 128, -54, -54), ("inner_product", 100, -70, -46), ("inner_product", 300, -60, -60),
    ("l2", 128, -54, -54), ("l2", 1536, -54.6, -54.6), ("l2", 1536, 44.5, -55), ("inner_product", 64, 30, -90),
    # (the last scales that take the pieces)
    ("l2", 96, -42, -42), ("l2", 96, 36, -42), ("inner_product", 96, -42, 36),
])
def test_scales_far_from_one(engine, oracle, metric, d, eb, eq):
    """Values whose two scales multiply to (or whose seeds are) past float32's
    range: sums that float32 holds, so the answers are ordinary ones.  A zero
    row, and one whose squares underflow."""
    r = np.random.default_rng(d)
    n, nq = size_of(d)
    base, q = rows_of("float", n, d, r), rows_of("float", nq, d, r)
    base *= np.float32(2.0 ** eb)
    q *= np.float32(2.0 ** eq)
    if metric == "l2" and eb < 0:
        base[7] = 0
        if eb == -54:
            base[8] *= np.float32(2.0 ** -20)
    check(engine, oracle, base, q, 10, metric, False)


@pytest.mark.parametrize("kind,d", [("bytes", 96), ("float", 96), ("outlier", 96),
                                    ("bytes", 131), ("float", 272), ("outlier", 272)])
def test_prefilter(engine, oracle, kind, d):
    r = np.random.default_rng(7)
    n, nq = size_of(d)
    base, q = rows_of(kind, n, d, r), rows_of(kind, nq, d, r)
    check(engine, oracle, base, q, 12, "l2", kind == "bytes", bitset=r.random(n) < 0.3)


@pytest.mark.parametrize("n,nq,d,k,metric", [
    (200_003, 513, 1536, 10, "inner_product"), (300_001, 2_003, 257, 10, "l2"),
    (150_037, 1_281, 800, 16, "inner_product"), (260_011, 1_500, 400, 40, "l2"),
    (2_999, 60_000, 860, 10, "l2"),
])
def test_binary16_deep_batches(engine, oracle, n, nq, d, k, metric):
    """The tile kernel on binary16 rows: its edges in rows, queries and dims."""
    r = np.random.default_rng(n + d)
    base = r.standard_normal((n, d), dtype=np.float32).astype(np.float16)
    q = r.standard_normal((nq, d), dtype=np.float32).astype(np.float16)
    check(engine, oracle, base, q, k, metric, False, count=8)


def test_binary16_deep_prefilter(engine, oracle):
    r = np.random.default_rng(8)
    base = r.standard_normal((240_001, 320), dtype=np.float32).astype(np.float16)
    q = r.standard_normal((2_001, 320), dtype=np.float32).astype(np.float16)
    check(engine, oracle, base, q, 20, "l2", False, count=8, bitset=r.random(len(base)) < 0.4)


def test_mixed_sides_and_ties(engine, oracle):
    """Integer rows against real queries (one side has lo pieces), and rows
    that repeat: the lowest ids come first."""
    r = np.random.default_rng(3)
    base = rows_of("bytes", N, 64, r)
    base[40_000:40_300] = base[100:400]
    q = rows_of("float", NQ, 64, r) + np.float32(100)
    check(engine, oracle, base, q, 10, "l2", False)
    q = base[100:100 + NQ].copy()
    check(engine, oracle, base, q, 10, "l2", True)


@pytest.mark.parametrize("value", [np.inf, -np.inf])
def test_infinite_values_take_the_float32_route(engine, oracle, value):
    r = np.random.default_rng(5)
    base, q = rows_of("float", N, 64, r), np.abs(rows_of("float", NQ, 64, r))
    base[123, 5] = value
    ids, dist = engine.brute_force_knn(base, q, 3, "inner_product")
    pick = sample(NQ)
    oi, od = oracle.knn(base, q[pick], 3, "inner_product")
    assert (ids[pick] == oi).mean() > 0.99
    if value > 0:
        assert (ids[:, 0] == 123).all() and np.isposinf(dist[:, 0]).all()
    else:
        assert not (ids == 123).any()


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("n,nq,d,k,metric", [
    (130, 5, 320, 10, "l2"), (20_003, 32, 257, 10, "cosine"), (5_001, 1, 1536, 16, "l2"),
    (9_999, 31, 500, 60, "l2"), (127, 8, 300, 3, "inner_product"), (12_345, 17, 640, 10, "cosine"),
])
def test_deep_rows_few_queries(engine, oracle, f16, n, nq, d, k, metric):
    """The row-split kernel: norms summed beside the products, partial tiles, a
    redo (k past the lists) that reads the norms it wrote, a zero row."""
    r = np.random.default_rng(n + d)
    base = r.standard_normal((n, d)).astype(np.float16 if f16 else np.float32)
    q = r.standard_normal((nq, d)).astype(base.dtype)
    base[n // 2] = 0
    if k > 16:  # more neighbours side by side than a list holds
        base[64:64 + k] = q[0] + (r.standard_normal((k, d)) * 0.1).astype(base.dtype)
    if metric == "cosine":
        base[n // 2] = base[n // 2 - 1]  # (the bound divides by the row's norm)
    check(engine, oracle, base, q, k, metric, False)


@pytest.mark.parametrize("kind", ["bytes", "normal", "outlier"])
@pytest.mark.parametrize("nq,k", [(1_025, 10), (2_000, 16)])
def test_routes_with_their_own_rounds(engine, oracle, kind, nq, k):
    """More queries than the bounded merge takes: the hi kernel's splits are
    finer than the other two routes', whose last segments stay empty."""
    r = np.random.default_rng(nq)
    base, q = rows_of(kind, N, 128, r), rows_of(kind, nq, 128, r)
    check(engine, oracle, base, q, k, "l2", kind == "bytes")


def held_after(engine, call):
    """Device memory that the engine keeps after one call on an empty workspace."""
    import ctypes

    from mlxvs_amd import _hip

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        _hip.check(_hip.lib().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)), "hipMemGetInfo")
        return a.value

    call()
    _hip.synchronize()
    engine.release_workspace()
    _hip.DeviceBuffer(1 << 20)  # (the runtime returns freed memory by the next allocation)
    before = free()
    call()
    _hip.synchronize()
    return before - free()


def test_workspace_is_what_the_call_takes(engine):
    """The pieces are as large as the rows and everything else is small: the
    call's room is made at once, for all of it, and not doubled on the way."""
    from mlxvs_amd import _hip

    n, nq, d, k = 1_000_000, 2_600, 128, 10
    base, q = _hip.DeviceBuffer(n * d * 4), _hip.DeviceBuffer(nq * d * 4)
    ids, dist = _hip.DeviceBuffer(nq * k * 4), _hip.DeviceBuffer(nq * k * 4)
    r = np.random.default_rng(0)
    x = r.standard_normal((n, d), np.float32)
    base.upload(x)
    q.upload(x[:nq])
    pieces = (n + nq) * d * 4
    held = held_after(engine, lambda: engine.brute_force_knn_device(
        base.value, n, q.value, nq, d, k, "l2", ids.value, dist.value))
    assert pieces <= held <= 1.25 * pieces
    lists = 512
    off = np.linspace(0, n, lists + 1).astype(np.int32)
    cen, offs, ind = (_hip.DeviceBuffer.from_array(a) for a in
                      (x[off[:-1]], off, np.arange(n, dtype=np.int32)))
    held = held_after(engine, lambda: engine.ivf_flat_search_device(
        cen.value, lists, base.value, n, ind.value, offs.value, d, "l2", q.value, nq, k,
        ids.value, dist.value, n_probes=16))
    assert pieces <= held <= 1.25 * pieces
    engine.release_workspace()
