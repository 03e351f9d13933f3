"""Bank updates: the placement kernel at the edges of its blocks (16 rows)
and slices (320 values), rows that are not finite, updates one after the
other without a wait, and refused updates that must leave the bank as it
was.  Ids and score bits equal the oracle's over the live rows."""

import numpy as np
import pytest

import oracle
from graftrepository_amd import MlaNodeBank
from graftrepository_amd.node_bank import as_bf16_bits, bf16_bits_to_f32

pytestmark = pytest.mark.gpu


def route_like_oracle(bank, live, q, k):
    res = bank.route(q, k, timed=False)
    ids = np.asarray(sorted(live), dtype=np.uint64)
    want, sc, _ = oracle.mla_route(np.stack([live[int(i)] for i in ids]), q, k, node_ids=ids)
    np.testing.assert_array_equal(res.ids, want)
    np.testing.assert_array_equal(res.scores.view(np.uint32), sc.view(np.uint32))


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("dim", [1, 7, 288, 319, 320, 321, 643])
@pytest.mark.parametrize("count", [1, 15, 16, 17, 200])
def test_placed_rows(hip_lib, count, dim, dtype):
    rng = np.random.default_rng(count * 1000 + dim)
    rows = rng.standard_normal((40 + count, dim)).astype(np.float32)
    rows[41 % len(rows)] = 0.0
    if count > 15:
        rows[50, dim // 2] = np.nan
        rows[54, 0] = np.inf
    bits = as_bf16_bits(rows) if dtype == "bf16" else rows
    values = bf16_bits_to_f32(bits).reshape(rows.shape) if dtype == "bf16" else rows
    q = rng.standard_normal((1, dim)).astype(np.float32)
    q_in = as_bf16_bits(q) if dtype == "bf16" else q
    q = bf16_bits_to_f32(q_in).reshape(q.shape) if dtype == "bf16" else q
    with MlaNodeBank(bits[:40], dtype=dtype, capacity=400) as bank:
        bank.evict(np.arange(3, 23, 2, dtype=np.uint64))  # holes the new rows fill first
        bank.append(bits[40:], np.arange(count, dtype=np.uint64) + 1000)
        res = bank.route(q_in, 16, timed=False)
    keep = [i for i in range(40) if not (3 <= i < 23 and i % 2)]
    ids = np.asarray(keep + list(range(1000, 1000 + count)), np.uint64)
    want, sc, _ = oracle.mla_route(values[keep + list(range(40, 40 + count))], q, 16, node_ids=ids)
    np.testing.assert_array_equal(res.ids, want)
    np.testing.assert_array_equal(res.scores.view(np.uint32), sc.view(np.uint32))


# 300 rows: one part; 2000 rows of 288: several parts; 9000: the copy engine
@pytest.mark.parametrize("count", [300, 2000, 9000])
def test_updates_back_to_back(hip_lib, count):
    rng = np.random.default_rng(count)
    dim, n = 288, 12_000
    rows = rng.standard_normal((n, dim)).astype(np.float32)
    q = rng.standard_normal((1, dim)).astype(np.float32)
    live = {i: rows[i] for i in range(n)}
    with MlaNodeBank(rows, capacity=n + 500) as bank:
        for step in range(4):
            out = rng.choice(sorted(live), size=count, replace=False).astype(np.uint64)
            new = np.concatenate([out[: count // 2], np.arange(count // 2, dtype=np.uint64)
                                  + 100_000 * (step + 1)])
            fresh = rng.standard_normal((new.size, dim)).astype(np.float32)
            bank.evict(out)
            bank.append(fresh, new)
            for i in out.tolist():
                del live[i]
            live.update(zip(new.tolist(), fresh))
        route_like_oracle(bank, live, q, 16)


def test_refused_updates_change_nothing(hip_lib):
    rng = np.random.default_rng(3)
    rows = rng.standard_normal((100, 32)).astype(np.float32)
    q = rng.standard_normal((1, 32)).astype(np.float32)
    live = {i: rows[i] for i in range(100)}
    with MlaNodeBank(rows, capacity=128) as bank:
        for ids in ([5, 7, 5], [5, 777]):
            with pytest.raises(RuntimeError):
                bank.evict(np.asarray(ids, np.uint64))
        for ids in ([200, 201, 200], [200, 5], [200, 2**64 - 1], list(range(200, 360))):
            with pytest.raises(RuntimeError):
                bank.append(np.zeros((len(ids), 32), np.float32), np.asarray(ids, np.uint64))
        route_like_oracle(bank, live, q, 16)
        # the ids the refused calls named are as free, or as live, as before
        bank.evict(np.asarray([5, 7], np.uint64))
        bank.append(rows[[7, 5, 0]], np.asarray([200, 5, 201], np.uint64))
        del live[7]
        live.update({5: rows[5], 200: rows[7], 201: rows[0]})
        assert bank.info()["live"] == len(live)
        route_like_oracle(bank, live, q, 16)
