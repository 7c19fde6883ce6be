"""Exact mode where the sums have to be done again in the CPU's order: products of very different size,
rows around the 64-dimension blocks of the wide form, more flagged candidates than it takes at a time,
and the narrow form, against the oracle (ids and distances bit for bit)."""
import numpy as np
import pytest

import pyoracle
import song_amd

pytestmark = pytest.mark.gpu


# dim 257 / 320 / 961: one past a unit boundary, whole blocks, a last block of one unit; 40 and 130: the
# narrow shapes (one lane per row); 1,030: the widest shape
@pytest.mark.parametrize("dim", [40, 130, 257, 320, 961, 1030])
@pytest.mark.parametrize("metric", ["l2", "ip", "cos"])
def test_sums_that_round_keep_the_cpu_order(dim, metric):
    rng = np.random.default_rng(dim)
    n, nq, pq = 600, 24, 40
    # values over 2^-20 .. 1: nearly every row has products below the sum's last bit
    scale = np.exp2(rng.integers(-20, 1, size=(n + nq, dim))).astype(np.float32)
    x = (rng.standard_normal((n + nq, dim)) * scale).astype(np.float32)
    base, query = x[:n], x[n:].copy()
    graph = pyoracle.build(base, metric)
    # a vertex with 31 neighbours: more than 16 candidates at once
    graph = graph.copy()
    graph[0, 0] = 31
    graph[0, 1:32] = np.arange(1, 32)
    ix = song_amd.Index(base, graph, metric)
    want, dist = pyoracle.search_batch(base, graph, metric, query, pq, threads=4)
    ids, ds, flags = ix.search(query, pq, pq, mode=song_amd.MODE_EXACT)
    assert np.array_equal(ids, want[:, :pq].astype(np.int64)) and not flags.any()
    assert np.array_equal(ds, dist[:, :pq].astype(np.float32))


def test_more_than_a_stage_of_front_entries():
    """A budget whose list is rebuilt from its front many times, with ids, distances and every counter
    of the first k equal to the oracle's order (vertices far from the query first)."""
    rng = np.random.default_rng(5)
    base = rng.integers(0, 200, size=(2500, 12)).astype(np.float32)
    query = rng.integers(0, 200, size=(40, 12)).astype(np.float32)
    graph = pyoracle.build(base, "l2")
    ix = song_amd.Index(base, graph, "l2")
    for pq in (63, 64, 65, 130, 700, 2400):
        want, _ = pyoracle.search_batch(base, graph, "l2", query, pq, threads=4)
        for bg in (0, 1):
            for mode in (song_amd.MODE_EXACT, song_amd.MODE_FP32):
                ids, _, flags = ix.search(query, pq, pq, mode=mode, best_in_global=bg)
                assert np.array_equal(ids, want[:, :pq].astype(np.int64)), (pq, bg, mode)


@pytest.mark.parametrize("bits", [16, 32])
def test_searches_that_outgrow_the_table(bits):
    """Small LDS tables push most vertices into the global one: same ids, no flag."""
    rng = np.random.default_rng(9)
    base = rng.standard_normal((6000, 24)).astype(np.float32)
    query = rng.standard_normal((50, 24)).astype(np.float32)
    graph = pyoracle.build(base, "l2")
    ix = song_amd.Index(base, graph, "l2")
    want, _ = pyoracle.search_batch(base, graph, "l2", query, 300, threads=4)
    for h in (8, 9, 11):
        ids, _, flags = ix.search(query, 300, 300, mode=song_amd.MODE_EXACT, hash_log2=h, visited_bits=bits, retry=0)
        assert np.array_equal(ids, want[:, :300].astype(np.int64)) and not flags.any()
