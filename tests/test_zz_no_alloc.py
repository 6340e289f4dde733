"""The no-allocation entry point (mlxvs_brute_force_knn_device_noalloc),
called through the C ABI, against mlxvs_brute_force_knn_device on the same
device inputs.  Integer rows: bit-identical ids and distances, also where the
allocating entry multiplies large float32 batches as binary16 pieces and this
one on the float32 MFMA (both sums are exact).  Real values in such batches
differ by rounding.  Calls in a row, later ones smaller (the shared scratch keeps the earlier
calls' contents), one with k = 64 (lists shorter than k, the merge's flags
and the redo of flagged queries all in the scratch), then the rejection of a
workspace beyond the fixed scratch, with device buffers of the real size.
"""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

INVALID = 1


def run(engine, fn, db, n, dq, nq, d, k, metric, f16=False):
    from mlxvs_amd import _hip

    di = _hip.DeviceBuffer(nq * k * 4)
    dd = _hip.DeviceBuffer(nq * k * 4)
    rc = fn(db.value, n, dq.value, nq, d, int(f16), k, int(metric), di.value, dd.value, None)
    return rc, di, dd


@pytest.mark.parametrize("f16", [False, True])
def test_no_alloc_matches_the_allocating_entry(engine, f16):
    from mlxvs_amd import _hip, synth

    lib = engine._L()
    # (at 300 and 500 queries, over 1,024 candidates a query, the allocating
    # entry merges by the bounded batch merge and the no-allocation entry by
    # the merge levels, so the comparison covers both; at k = 64 the redo
    # flags as well)
    cases = [(200_000, 2_000, 128, 10, engine.Metric.l2),
             (30_000, 300, 64, 8, engine.Metric.inner_product),
             (50_000, 500, 128, 64, engine.Metric.l2)]
    for n, nq, d, k, metric in cases:
        print(f"[no_alloc] f16={f16} n={n} nq={nq} d={d} k={k} metric={int(metric)}", flush=True)
        cen = synth.c2_centres()
        base = synth.c2_rows(1, 0, n, centres=cen)[:, :d]
        q = synth.c2_rows(2, 0, nq, centres=cen)[:, :d]
        if f16:
            base, q = base.astype(np.float16), q.astype(np.float16)
        db = _hip.DeviceBuffer.from_array(np.ascontiguousarray(base))
        dq = _hip.DeviceBuffer.from_array(np.ascontiguousarray(q))
        rc, wi, wd = run(engine, lib.mlxvs_brute_force_knn_device, db, n, dq, nq, d, k, metric,
                         f16)
        assert rc == 0, lib.mlxvs_last_error()
        rc, gi, gd = run(engine, lib.mlxvs_brute_force_knn_device_noalloc, db, n, dq, nq, d, k,
                         metric, f16)
        assert rc == 0, lib.mlxvs_last_error()
        _hip.synchronize()
        want_i, want_d = wi.download((nq, k), np.int32), wd.download((nq, k), np.float32)
        got_i, got_d = gi.download((nq, k), np.int32), gd.download((nq, k), np.float32)
        assert np.array_equal(got_i, want_i)
        assert np.array_equal(got_d.view(np.uint32), want_d.view(np.uint32))


@pytest.mark.parametrize("metric", ["l2", "inner_product"])
def test_large_real_batches_differ_by_rounding(engine, metric):
    """The allocating entry takes the two binary16 pieces here, this one the
    float32 kernels: each list's distances agree, place by place, within twice
    one distance's error, and so do the rows' own distances in 64 bits.  In units
    of 2^-24 of sum |q_i b_i| <= |q||b| a product's sum is off by at most d + 9
    (either unit); L2 takes that twice, and d + 4 of |q|^2 + |b|^2."""
    from mlxvs_amd import _hip

    lib = engine._L()
    n, nq, d, k = 120_011, 1_203, 128, 10
    r = np.random.default_rng(4)
    base, q = (r.standard_normal((m, d), np.float32) for m in (n, nq))
    db, dq = _hip.DeviceBuffer.from_array(base), _hip.DeviceBuffer.from_array(q)
    lists = []
    for fn in (lib.mlxvs_brute_force_knn_device, lib.mlxvs_brute_force_knn_device_noalloc):
        rc, di, dd = run(engine, fn, db, n, dq, nq, d, k, engine.Metric[metric])
        assert rc == 0, lib.mlxvs_last_error()
        _hip.synchronize()
        lists.append((di.download((nq, k), np.int32), dd.download((nq, k), np.float32)))
    bn, qn = np.linalg.norm(base, axis=1).max(), np.linalg.norm(q, axis=1)[:, None]
    err = (d + 9) * 2.0 ** -24 * qn * bn
    if metric == "l2":
        err = 2 * err + (d + 4) * 2.0 ** -24 * (qn ** 2 + bn ** 2)
    own = []
    for ids, dist in lists:
        b, x = base[ids].astype(np.float64), q[:, None].astype(np.float64)
        own.append(((b - x) ** 2).sum(2) if metric == "l2" else (b * x).sum(2))
        assert (np.abs(dist - own[-1]) <= err).all()
    assert (np.abs(lists[0][1].astype(np.float64) - lists[1][1]) <= 2 * err).all()
    assert (np.abs(own[0] - own[1]) <= 4 * err).all()
    assert not np.array_equal(lists[0][1], lists[1][1])  # (two routes, not one)


def test_no_alloc_rejects_what_it_cannot_hold(engine):
    from mlxvs_amd import _hip

    lib = engine._L()
    fn = lib.mlxvs_brute_force_knn_device_noalloc
    n, d = 1_000_000, 4
    db = _hip.DeviceBuffer.from_array(np.zeros((n, d), np.float32))
    # 100,000 queries' lists need more than the 64 MiB of scratch
    nq = 100_000
    dq = _hip.DeviceBuffer.from_array(np.zeros((nq, d), np.float32))
    rc, _, _ = run(engine, fn, db, n, dq, nq, d, 10, engine.Metric.l2)
    assert rc == INVALID and b"MiB of scratch" in lib.mlxvs_last_error()
    _hip.synchronize()
