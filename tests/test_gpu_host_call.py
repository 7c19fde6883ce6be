"""The host-buffer search through its kept workspaces: pinned copies, plain copies and calls larger
than the pool keeps, in every arithmetic mode, and from several threads at once."""
import threading

import numpy as np
import pytest

import pyoracle
import song_amd
from song_amd import datasets

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def index():
    base, query = datasets.mixture_l2(n_base=3000, n_query=9000, dim=64, n_centers=30, seed=21)
    return song_amd.Index(base, pyoracle.build(base, "l2"), "l2"), base, query


def _device(ix, q, pq, k, mode):
    import torch

    qd = torch.from_numpy(q).cuda()
    ids = torch.empty((len(q), k), dtype=torch.int32, device="cuda")
    ds = torch.empty((len(q), k), device="cuda")
    ix.search_device(qd, pq, k, ids, ds, mode=mode)
    return ids.cpu().numpy().astype(np.int64), ds.cpu().numpy()


# one query; the last call with pinned copies (k 20: 420 bytes a query, 1 MB = 2,496) and the first
# without; a workspace above the 8 MB that the pool keeps
@pytest.mark.parametrize("nq,k", [(1, 1), (5, 20), (2400, 20), (2600, 20), (9000, 100)])
@pytest.mark.parametrize("whole", [True, False])
def test_host_call_equals_device_call(index, nq, k, whole):
    ix, _, query = index
    q = query[:nq] if whole else query[:nq] + np.float32(0.25)
    want_i, want_d = _device(ix, q, 100, k, song_amd.MODE_AUTO)
    for _ in range(2):  # a new workspace, then a kept one
        ids, ds, flags = ix.search(q, 100, k)
        assert np.array_equal(ids, want_i) and np.array_equal(ds, want_d) and not flags.any()


def test_columns_past_pq_are_padding(index):
    ix, _, query = index
    ids, ds, _ = ix.search(query[:7], 5, 5)
    wide = np.empty((7, 9), dtype=np.uint64)
    dist = np.empty((7, 9), dtype=np.float32)
    o = song_amd.make_opts()
    q = np.ascontiguousarray(query[:7])
    import ctypes

    song_amd._check(song_amd.lib().song_search(ix._h, song_amd._ptr(q), 7, 5, 9, song_amd._ptr(wide), song_amd._ptr(dist),
                                               None, ctypes.byref(o)))
    assert np.array_equal(wide[:, :5].astype(np.int64), ids) and np.array_equal(dist[:, :5], ds)
    assert (wide[:, 5:] == np.uint64(0xFFFFFFFFFFFFFFFF)).all() and np.isinf(dist[:, 5:]).all()


def test_calls_from_several_threads(index):
    ix, _, query = index
    parts = [query[i * 300:(i + 1) * 300] for i in range(6)]
    want = [ix.search(p, 64, 10)[0] for p in parts]
    got = [None] * 6

    def work(i):
        for _ in range(4):
            got[i] = ix.search(parts[i], 64, 10)[0]

    ts = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
