"""Options of a call at sizes that the four-cells-per-wave kernel takes (launches
of more than 6144 cells), against the CPU oracle: ragged initial guesses with
empty rows, hidden cells, duplicates, leaf sizes, no pre-clip; and the rows of
guesses of the lane-per-query search on clustered points.  Whole-number outputs:
no tolerance (distances: 2e-6, as for the other searches)."""
import numpy as np
import pytest

from paragram_amd import workloads
from tests.test_gpu_knn_guesses import check_rows, guesses
from tests.test_gpu_parity import assert_matches_oracle, run

pytestmark = pytest.mark.gpu
N = 9001


def weights(n, top, seed):
    return np.random.default_rng(seed).uniform(0, top, n).astype(np.float32)


@pytest.mark.parametrize("weighted", [False, True])
def test_ragged_guesses(gpu, weighted):
    import torch

    print(f"main kernel: ragged guesses, weighted {weighted}", flush=True)
    pts = workloads.uniform(N, 21)
    w = weights(N, 2e-3, 22) if weighted else None
    adj, off, _ = run(gpu, pts, w)
    rng = np.random.default_rng(23)
    rows = []
    for i in range(N):
        kind = rng.integers(5)
        row = adj[off[i]:off[i + 1]]
        if kind == 0:
            row = row[:0]  # empty
        elif kind == 1:
            row = rng.integers(-1, N, rng.integers(1, 40))  # anything, repeats and -1 among them
        elif kind == 2:
            row = np.concatenate([row, row, [i]])  # twice, and the point itself
        elif kind == 3:
            row = rng.permutation(row)[: len(row) // 2]
        rows.append(row.astype(np.int32))
    g = torch.from_numpy(np.concatenate(rows)).to(gpu)
    o = torch.from_numpy(np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)).to(gpu)
    assert_matches_oracle(run(gpu, pts, w, initial_guesses=g, initial_guesses_offsets=o), pts, w)


@pytest.mark.parametrize("top", [1e-4, 6e-3])
def test_hidden_cells(gpu, top):
    print(f"main kernel: weights up to {top}", flush=True)
    pts, w = workloads.uniform(N, 31), weights(N, top, 32)
    got = run(gpu, pts, w)
    assert_matches_oracle(got, pts, w)
    assert top < 1e-3 or (got[2] == 3).sum() > N // 10


@pytest.mark.parametrize("weighted", [False, True])
def test_duplicates(gpu, weighted):
    print(f"main kernel: duplicates, weighted {weighted}", flush=True)
    pts = workloads.uniform(N, 41)
    pts = np.concatenate([pts, pts[:700], pts[:90], pts[:90]])
    w = None
    if weighted:  # some copies weigh the same, some do not
        w = weights(N, 1e-3, 42)
        w = np.concatenate([w, w[:700], 0.5 * w[:90], w[:90]]).astype(np.float32)
    assert_matches_oracle(run(gpu, pts, w), pts, w)


@pytest.mark.parametrize("leaf,knn", [(1, 8), (5, 8), (32, 8), (32, 0)])
def test_leaf_sizes_and_no_preclip(gpu, leaf, knn):
    print(f"main kernel: leaf size {leaf}, knn {knn}", flush=True)
    pts = workloads.uniform(N, 51)
    assert_matches_oracle(run(gpu, pts, leaf_size=leaf, knn=knn), pts)


@pytest.mark.parametrize("k", [16, 5])
def test_lane_search_on_clusters(gpu, k):
    n = (3 << 16) + 1
    print(f"lane-per-query search: {n} clustered points, k={k}", flush=True)
    r = np.random.default_rng(61)
    c = r.random((64, 3))
    pts = np.concatenate([c[r.integers(0, 64, n // 2)] + 0.003 * r.standard_normal((n // 2, 3)), r.random((n - n // 2, 3))])
    pts = pts[r.permutation(n)].astype(np.float32)
    ids, d2, _ = guesses(gpu, pts, k)
    check_rows(ids, k)
    # rows come in the index's order: the K-th distances as a sorted list against those of a sample of queries
    p = pts.astype(np.float64)
    pick = r.permutation(n)[:200]
    want = np.sort(((p[pick, None, :] - p[None, :, :]) ** 2).sum(-1), axis=1)[:, k]
    have = np.sort(d2.astype(np.float64))
    at = np.clip(np.searchsorted(have, want), 1, n - 1)
    near = np.minimum(np.abs(have[at] - want), np.abs(have[at - 1] - want))
    assert (near <= 2e-6 * want).all()
