"""The single-query MLA kernel's forms and the wave-wide top-k list, at the
sizes where they change: tiles per compute unit (deep form to 8, then 16
waves, then several rounds), chunks per row against the load batches, and
tiles that bring many candidates or ties at once.  Ids and score bits equal
the oracle's (exact by construction: the same fp64 operations in order)."""

import numpy as np
import pytest

import oracle
from graftrepository_amd import MlaNodeBank, workloads as wl

pytestmark = pytest.mark.gpu


def check(rows, qs, k, node_ids=None, dtype="f32"):
    with MlaNodeBank(rows, node_ids, dtype=dtype) as bank:
        res = bank.route(qs, k, timed=False)
        timed = bank.route(qs, k)
    as_f32 = rows if dtype == "f32" else (rows.astype(np.uint32) << 16).view(np.float32)
    q32 = qs if dtype == "f32" else (qs.astype(np.uint32) << 16).view(np.float32)
    ids, sc, _ = oracle.mla_route(as_f32, q32, k, node_ids=node_ids)
    for r in (res, timed):
        np.testing.assert_array_equal(r.ids, ids)
        np.testing.assert_array_equal(r.scores.view(np.uint32), sc.view(np.uint32))


# one tile, a tile and a row, 1 and 2 tiles per CU, the deep form's last
# size, the first after it, two and four rounds of 16 waves (256 CUs)
@pytest.mark.parametrize("nodes", [1, 64, 65, 256 * 64, 256 * 64 + 1, 8 * 256 * 64,
                                   8 * 256 * 64 + 1, 16 * 256 * 64 + 700, 49 * 256 * 64])
def test_bank_sizes(hip_lib, nodes):
    rows, qs = wl.mla_rows(nodes, 12, seed=nodes), wl.mla_queries(2, 12, seed=nodes)
    check(rows, qs, min(5, nodes))


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("nodes", [3_000, 140_000])  # deep, 16 waves
@pytest.mark.parametrize("dim", [2, 47, 64, 71, 72, 73, 145])
def test_row_lengths(hip_lib, dim, nodes, dtype):
    check(wl.mla_rows(nodes, dim, seed=dim, dtype=dtype),
          wl.mla_queries(1, dim, seed=dim, dtype=dtype), 3, dtype=dtype)


@pytest.mark.parametrize("k", [1, 2, 15, 16])
@pytest.mark.parametrize("order", ["rising", "falling", "few values", "one value"])
def test_candidates_arrive_at_once(hip_lib, order, k):
    n = 2_000
    t = {"rising": np.arange(n), "falling": -np.arange(n), "few values": np.arange(n) % 5,
         "one value": np.zeros(n)}[order] / n
    rows = np.stack([np.cos(1 - t), np.sin(1 - t)], axis=1).astype(np.float32)
    ids = np.random.default_rng(k).permutation(n).astype(np.uint64) + 7
    check(rows, np.array([[1.0, 0.0]], np.float32), k, node_ids=ids)
