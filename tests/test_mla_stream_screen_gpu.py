"""The stream screen (fp32 banks, and bf16 rows and passes that the ring
screen does not take): ids and score bits against the oracle at the edges of
its batches, column tiles and tiles per sub-stream, and its bound held pair
by pair.

The oracle scores in fp64 and the library rescores every candidate in fp64,
so results are compared bit for bit."""

import numpy as np
import pytest

import oracle
from graftrepository_amd import MlaNodeBank, workloads as wl
from graftrepository_amd.node_bank import as_bf16_bits, bf16_bits_to_f32
from tests.test_screen_bound_gpu import cancelling, mla_queries, mla_rows, spread

pytestmark = pytest.mark.gpu


def f32_of(x):
    return bf16_bits_to_f32(x).reshape(x.shape) if x.dtype == np.uint16 else x


def check(bank, rows, qs, k, node_ids=None, query_dtype="f32"):
    res = bank.route(qs, k, query_dtype=query_dtype)
    ids, sc, _ = oracle.mla_route(f32_of(rows), f32_of(qs), k, node_ids=node_ids)
    np.testing.assert_array_equal(res.ids, ids)
    np.testing.assert_array_equal(res.scores.view(np.uint32), sc.view(np.uint32))


# rows of one value up to ones whose queries fill LDS 32 at a time; 1300
# values take the single-query kernel
@pytest.mark.parametrize("dim", [1, 17, 64, 65, 100, 144, 145, 280, 288, 300, 576, 1000, 1300])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_row_lengths(hip_lib, dim, dtype):
    rows = wl.mla_rows(3001, dim, seed=dim, dtype=dtype)
    qs = wl.mla_queries(40, dim, seed=dim)
    with MlaNodeBank(rows, dtype=dtype) as bank:
        check(bank, rows, qs, 6)
        stats = bank.route_stats()
    assert stats["batched"] == (0 if (dtype, dim) == ("f32", 1300) else 40)
    if 64 <= dim <= 576:
        # A tile keeps two entries per query; three of its 32 rows near the
        # sixth best of 3,001 take the exact path.  About 1e-2 a call.
        assert stats["fallbacks"] <= 2


# Column tiles and passes; one tile up to several tiles per sub-stream.  The
# results compared are to come from the screen and the merge: a tile keeps
# two entries per query, so one or two tiles certify up to two results; at
# 2,000 rows and k = 16 a tenth of the queries have three in one tile.
@pytest.mark.parametrize("nq,k", [(4, 1), (32, 3), (33, 16), (64, 8), (65, 5), (128, 2), (130, 7)])
@pytest.mark.parametrize("n", [20, 32, 33, 2000, 70_001])
def test_query_counts(hip_lib, nq, k, n):
    rows = wl.mla_rows(n, 96, seed=n)
    qs = wl.mla_queries(nq, 96, seed=n + 1)
    with MlaNodeBank(rows) as bank:
        check(bank, rows, qs, k if n >= 2000 else min(k, 2))
        stats = bank.route_stats()
        assert stats["batched"] == nq and stats["fallbacks"] <= nq // 4


# The ring screen's runs: none, one or several tiles each, with k that a lane
# half's two entries per tile certify for nearly every query
@pytest.mark.parametrize("n,k", [(20, 2), (33, 2), (600, 8), (1000, 12), (5000, 16), (32_768, 16), (33_001, 16),
                                 (100_003, 16)])
def test_ring_runs(hip_lib, n, k):
    rows = wl.mla_rows(n, 72, seed=n, dtype="bf16")
    qs = wl.mla_queries(200, 72, seed=n + 1, dtype="bf16")
    with MlaNodeBank(rows, dtype="bf16") as bank:
        check(bank, rows, qs, k, query_dtype="bf16")
        stats = bank.route_stats()
        assert stats["batched"] == 200 and stats["fallbacks"] <= 20


# Calls that the screen would send back to the single-query kernel take that
# at once: too few entries for k, or most queries with three in one tile
@pytest.mark.parametrize("n,k,nq,batched", [
    (20, 3, 64, False), (300, 16, 64, False), (1000, 16, 3, False), (1000, 16, 8, True),
    (2000, 16, 3, True), (1000, 3, 2, False), (1000, 3, 3, True), (9000, 3, 2, True)])
def test_which_calls_are_batched(hip_lib, n, k, nq, batched):
    rows, qs = wl.mla_rows(n, 96, seed=n), wl.mla_queries(nq, 96, seed=n + 1)
    with MlaNodeBank(rows) as bank:
        check(bank, rows, qs, k)
        stats = bank.route_stats()
    assert stats["batched"] == (nq if batched else 0)
    assert stats["single"] == (stats["fallbacks"] if batched else nq)


def test_churn_warmup_and_bf16_queries(hip_lib):
    rng = np.random.default_rng(3)
    rows = wl.mla_rows(5000, 280, seed=5)
    ids = np.arange(5000, dtype=np.uint64) * 2 + 1
    qs = wl.mla_queries(24, 280, seed=5)
    with MlaNodeBank(rows, ids, capacity=6000) as bank:
        gone = rng.choice(5000, size=400, replace=False)
        bank.evict(ids[gone])
        fresh = wl.mla_rows(300, 280, seed=6)
        bank.append(fresh, np.arange(300, dtype=np.uint64) + 50_000)
        live = np.ones(5000, bool)
        live[gone] = False
        mat = np.concatenate([rows[live], fresh])
        node_ids = np.concatenate([ids[live], np.arange(300, dtype=np.uint64) + 50_000])
        check(bank, mat, qs, 8, node_ids)
        check(bank, mat, as_bf16_bits(qs), 8, node_ids, query_dtype="bf16")
        want, sc, _ = oracle.mla_route(mat, qs, 8, node_ids=node_ids)
        for timed in (True, False):
            r = bank.route(qs, 8, warmup=7, timed=timed)
            np.testing.assert_array_equal(r.ids, want)
            np.testing.assert_array_equal(r.scores.view(np.uint32), sc.view(np.uint32))
            assert np.isnan(r.device_ms) != timed
            assert 0.0 < bank.screen_ms() < 50.0
            if timed:
                assert bank.screen_ms() <= r.device_ms


def test_rows_the_screen_cannot_certify(hip_lib):
    # ties, zero, NaN and infinite rows, rows near the largest finite value
    # (their bf16 rounding overflows), all scores negative, empty queries
    rng = np.random.default_rng(8)
    base = rng.standard_normal((60, 128)).astype(np.float32)
    rows = np.repeat(base, 20, axis=0)
    rows[5] = 0.0
    rows[17, 3] = np.nan
    rows[21, 3] = np.inf
    qs = np.concatenate([base[:12] + 0.1 * base[12:24], np.zeros((1, 128), np.float32)]).astype(np.float32)
    qs[3, 0] = np.nan
    ids = rng.permutation(rows.shape[0]).astype(np.uint64) + 7
    with MlaNodeBank(rows, ids) as bank:
        check(bank, rows, qs, 10, ids)
    rows = rng.standard_normal((3000, 64)).astype(np.float32)
    rows[7] = np.float32(3.4e38) * np.sign(rows[7])
    qs = rng.standard_normal((8, 64)).astype(np.float32) * np.float32(2.0 ** -20)
    qs[1] = np.sign(rows[7])
    with MlaNodeBank(rows) as bank:
        check(bank, rows, qs, 6)
    rows, qs = np.abs(rows[8:]), -np.abs(qs)
    with MlaNodeBank(rows) as bank:
        check(bank, rows, qs, 6)


# the stream screen's column tiles, and the ring (200 bf16 queries)
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("nq", [2, 3, 40, 200])
@pytest.mark.parametrize("dim", [64, 600])
def test_rows_whose_norm_overflows(hip_lib, dim, nq, dtype):
    # Four rows that score 0 by the law (an infinite norm) in one tile with
    # some queries' best row: their screened values are NaN and must not
    # push that row out.  Slots 1, 2, 9 and 18 share a lane half with 10, 11
    # and 16, 17.
    rng = np.random.default_rng(nq + dim)
    rows = rng.standard_normal((9000, dim)).astype(np.float32)
    qs = rng.standard_normal((nq, dim)).astype(np.float32)
    for slot, query in zip((10, 11, 16, 17), range(nq)):
        rows[slot] = qs[query] + 0.1 * rows[slot]
    for slot in (1, 2, 9, 18):
        rows[slot] = np.float32(3.38e38 if dtype == "bf16" else 3.4e38) * np.sign(rows[slot])
    bits = as_bf16_bits(rows) if dtype == "bf16" else rows
    qb = as_bf16_bits(qs) if dtype == "bf16" else qs
    with MlaNodeBank(bits, dtype=dtype) as bank:
        check(bank, bits, qb, 6, query_dtype=dtype)
        assert bank.route_stats()["batched"] == nq


@pytest.mark.parametrize("adversarial", [False, True])
@pytest.mark.parametrize("count,dim", [(80, 288), (30, 570)])
def test_fp32_screen_obeys_its_bound(hip_lib, adversarial, count, dim):
    rng = np.random.default_rng(31 + adversarial)
    n = 2048
    fam = np.array_split(np.arange(n), 6 if adversarial else 3)
    rows = np.empty((n, dim))
    rows[fam[0]] = rng.standard_normal((fam[0].size, dim))
    rows[fam[1]] = spread(rng, (fam[1].size, dim), -40, 40)
    rows[fam[2]] = cancelling(rng, (fam[2].size, dim), 2.0 ** -18)
    if adversarial:
        rows[fam[3]] = spread(rng, (fam[3].size, dim), -145, -118)  # subnormals included
        rows[fam[4]] = spread(rng, (fam[4].size, dim), 90, 110)
        rows[fam[5]] = rng.standard_normal((fam[5].size, dim))
        rows[fam[5][::7]] = 0.0
    rows = rows.astype(np.float32)
    q = mla_queries(rng, count, dim)
    with MlaNodeBank(rows) as bank:
        vals, bounds, ids = bank.probe_screen(q, query_dtype="f32")
    score = oracle.mla_scores(rows, q)
    norms = oracle.mla_row_norms(rows).astype(np.float64)
    nmax = norms[np.isfinite(norms)].max()
    big = np.array([oracle.mla_qnorm(x) for x in q]) * nmax
    assert np.all(np.isfinite(bounds[big < 2.0 ** 124]))
    assert np.all(np.isinf(bounds[big > 2.0 ** 126]))
    fin = np.isfinite(bounds)
    err = np.abs(vals[fin].astype(np.float64) - score[fin].astype(np.float64))
    ratio = err / bounds[fin, None]
    assert np.all(ratio <= 1.0), f"worst |s~ - score| / B = {ratio.max():.3g}"
    if not adversarial:
        # Gaussian queries: a far tighter bound than one bf16 rounding's 2^-8
        assert np.all(bounds[: count // 5] < 2.0 ** -10)
        assert ratio.max() > 1e-3


@pytest.mark.parametrize("count,dim", [(80, 570), (30, 300)])
def test_long_bf16_rows_obey_the_bound(hip_lib, count, dim):
    rng = np.random.default_rng(41)
    bits = mla_rows(rng, 2048, dim, True)
    q = mla_queries(rng, count, dim)
    with MlaNodeBank(bits, dtype="bf16") as bank:
        vals, bounds, _ = bank.probe_screen(q, query_dtype="f32")
    score = oracle.mla_scores(bf16_bits_to_f32(bits), q)
    fin = np.isfinite(bounds)
    assert fin.sum() >= count // 2
    err = np.abs(vals[fin].astype(np.float64) - score[fin].astype(np.float64))
    assert np.all(err <= bounds[fin, None])
