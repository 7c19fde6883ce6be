"""The default visited table around the lines of its size rules: a call's ids, distances and flags are
those of explicit table sizes, whatever the number of queries, the rows and the budget."""
import numpy as np
import pytest
import torch

import pyoracle
import song_amd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[(13, "cos"), (32, "l2"), (100, "ip")], ids=str)
def held(request):
    dim, metric = request.param
    rng = np.random.default_rng(dim)
    base = rng.standard_normal((4000, dim)).astype(np.float32)
    graph = pyoracle.build(base, metric)
    ix = song_amd.Index(base, graph, metric)
    ix.add_storage(song_amd.STORE_FP8)
    return ix, torch.from_numpy(rng.standard_normal((6200, dim)).astype(np.float32)).cuda(), base, graph, metric


# 2816 | 2817: where a 4 KB front stops fitting 11 waves a CU; 4096 | 4097: the 16 waves of 2^12 slots;
# 6200: more than 20 waves a CU
@pytest.mark.parametrize("nq,pq", [(1, 100), (2816, 256), (2817, 256), (2817, 512), (4096, 100), (4097, 100),
                                   (4097, 128), (4097, 129), (6200, 16), (6200, 128)])
@pytest.mark.parametrize("mode,storage", [(song_amd.MODE_EXACT, song_amd.STORE_F32),
                                          (song_amd.MODE_FP32, song_amd.STORE_F32),
                                          (song_amd.MODE_FP32, song_amd.STORE_FP8)])
def test_results_do_not_depend_on_the_table(held, nq, pq, mode, storage):
    ix, q, base, graph, metric = held
    got = []
    for hlog, noalloc in ((0, False), (12, False), (13, False), (0, True)):
        ids = torch.full((nq, 10), -7, dtype=torch.int32, device="cuda")
        ds = torch.full((nq, 10), -7.0, device="cuda")
        fl = torch.full((nq,), 99, dtype=torch.int32, device="cuda")
        if noalloc:
            song_amd.search_device_noalloc(ix, q[:nq], pq, 10, ids, ds, fl, mode=mode, storage=storage)
        else:
            ix.search_device(q[:nq], pq, 10, ids, ds, fl, mode=mode, storage=storage, retry=0, hash_log2=hlog)
        torch.cuda.synchronize()
        got.append((ids.cpu().numpy(), ds.cpu().numpy(), fl.cpu().numpy()))
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b)
    assert not got[0][2].any()
    if mode == song_amd.MODE_EXACT:
        want, dist = pyoracle.search_batch(base, graph, metric, q[:nq].cpu().numpy()[-50:], pq, threads=4)
        assert np.array_equal(got[0][0][-50:], want[:, :10])
        assert np.array_equal(got[0][1][-50:], dist[:, :10].astype(np.float32))
