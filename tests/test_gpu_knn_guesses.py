"""Rows of guesses (the diagram's pre-clip) against brute force in float64 and,
at the size where the lane-per-query search takes over, against that search:
the K-th squared distances (as a sorted list: rows come in the index's order),
and rows of distinct ids, short ones padded.  Tolerance: a squared distance of
float32 coordinates is three differences, squares and sums, each rounded to
2^-24 and under five roundings deep, so within 4e-7 of the exact one,
relatively; 2e-6 as for the lane-per-query search."""
import ctypes

import numpy as np
import pytest

from paragram_amd import workloads
from tests.test_gpu_wide import chain

pytestmark = pytest.mark.gpu
FLT_MAX = float(np.finfo(np.float32).max)


def guesses(gpu, pts, k):
    import torch

    from paragram_amd import _backend, _engine

    lib, p, n = _backend._C.lib, _engine._p, pts.shape[0]
    P = torch.from_numpy(np.ascontiguousarray(pts)).to(gpu)
    sp = ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)
    ws_bytes = lib.u64("pg_index_workspace_bytes", n)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=gpu)
    lib.call("pg_build_index", n, p(P), None, -1, p(ws), ws_bytes, sp)
    ids = torch.empty((n, k), dtype=torch.int32, device=gpu)
    d2 = torch.empty(n, dtype=torch.float32, device=gpu)
    lib.call("pg_knn_guesses", n, p(ws), 0, k, p(ids), p(d2), sp)
    all_ids, all_d2 = _engine.knn(lib, P, k)
    return ids.cpu().numpy(), d2.cpu().numpy(), all_d2.cpu().numpy()[:, k - 1]


def check_rows(ids, k):
    n = ids.shape[0]
    assert ((ids >= 0) & (ids < n)).all()
    full = np.sort(ids, axis=1)
    if n > k:
        assert (np.diff(full, axis=1) > 0).all(), "an id twice in a row"
        assert (ids != np.arange(n)[:, None]).all(), "a point is its own neighbour"


@pytest.mark.parametrize("k", [16, 5])
@pytest.mark.parametrize("n", [1, 2, 5, 6, 16, 17, 32, 33, 300, 3000, "chain"])
def test_guesses_match_brute_force(gpu, n, k):
    print(f"guesses n={n} k={k}", flush=True)
    pts = chain(20, 300) if n == "chain" else workloads.uniform(n, 50 + n)
    ids, d2, _ = guesses(gpu, pts, k)
    check_rows(ids, k)
    p = pts.astype(np.float64)
    dd = ((p[:, None, :] - p[None, :, :]) ** 2).sum(-1)
    np.fill_diagonal(dd, np.inf)
    want = np.sort(dd, axis=1)[:, k - 1] if p.shape[0] > k else np.full(p.shape[0], FLT_MAX)
    assert np.allclose(np.sort(d2.astype(np.float64)), np.sort(want), rtol=2e-6, atol=0)


@pytest.mark.parametrize("n", [(3 << 16) - 1, 3 << 16, (3 << 16) + 1])
def test_guesses_match_the_lane_search(gpu, n):
    print(f"guesses n={n}", flush=True)
    ids, d2, want = guesses(gpu, workloads.uniform(n, 9), 16)
    check_rows(ids, 16)
    assert np.allclose(np.sort(d2.astype(np.float64)), np.sort(want.astype(np.float64)), rtol=2e-6, atol=0)
