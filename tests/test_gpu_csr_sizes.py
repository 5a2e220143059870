"""The offsets' scan at the edges of its one-launch form, and the symmetry
check and row emission over rows around the lanes that share one, against
numpy.  Whole numbers: no tolerance."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def handles(gpu):
    import torch

    from paragram_amd import _backend, _engine

    return torch, _backend._C.lib, _engine, ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)


@pytest.mark.parametrize("n", [1, 2, 1023, 8191, 8192, 8193, 16383, 16384, 16385, 70000])
def test_scan(gpu, n):
    print(f"scan n={n}", flush=True)
    torch, lib, eng, sp = handles(gpu)
    counts = np.random.default_rng(n).integers(0, 50, n).astype(np.int32)
    c = torch.from_numpy(counts).to(gpu)
    out = torch.full((n + 1,), -1, dtype=torch.int32, device=gpu)
    tmp = torch.empty(max(lib.u64("pg_scan_tmp_bytes", n + 1), 4), dtype=torch.uint8, device=gpu)
    lib.call("pg_scan_counts", n, eng._p(c), eng._p(out), eng._p(tmp), sp)
    assert np.array_equal(out.cpu().numpy(), np.concatenate([[0], np.cumsum(counts)]))


@pytest.mark.parametrize("n,degree", [(2, 1), (40, 15), (41, 16), (42, 17), (60, 33), (700, 20)])
def test_symmetry_and_emission(gpu, n, degree):
    """Random rows of up to ``degree`` entries (some empty, stored in the index's
    order with gaps), the missing reverse edges and the entries at empty cells
    counted as numpy counts them, and the rows emitted in original order."""
    print(f"rows n={n} degree={degree}", flush=True)
    torch, lib, eng, sp = handles(gpu)
    rng = np.random.default_rng(n)
    # points on a line: the index's order is that of x
    x = rng.permutation(n).astype(np.float32)
    pts = torch.from_numpy(np.stack([x, 0 * x, 0 * x], 1)).to(gpu)
    ws_bytes = lib.u64("pg_index_workspace_bytes", n)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=gpu)
    lib.call("pg_build_index", n, eng._p(pts), None, -1, eng._p(ws), ws_bytes, sp)
    counts = rng.integers(1, degree + 1, n).astype(np.int32)
    counts[:: 7] = degree
    if n > 2:
        counts[3::11] = 0
    rows = [np.sort(rng.choice(np.delete(np.arange(n), u), counts[u], replace=False)).astype(np.int32)
            for u in range(n)]
    stride = degree + 3
    src = np.full((n, stride), -7, np.int32)
    for at, u in enumerate(np.argsort(x)):
        src[at, : counts[u]] = rows[u]
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    c, s, o = (torch.from_numpy(np.ascontiguousarray(a)).to(gpu) for a in (counts, src, offsets))
    stats = torch.zeros(eng.NUM_STATS, dtype=torch.int64, device=gpu)
    lib.call("pg_check_symmetry", n, eng._p(ws), eng._p(c), eng._p(s), None, stride, eng._p(o), eng._p(stats), sp)
    adj = torch.full((int(offsets[-1]),), -1, dtype=torch.int32, device=gpu)
    lib.call("pg_emit_csr", n, eng._p(ws), eng._p(c), eng._p(o), eng._p(s), None, stride, eng._p(adj), sp)
    assert np.array_equal(adj.cpu().numpy(), np.concatenate(rows))
    sets = [set(r.tolist()) for r in rows]
    dropped = sum(counts[v] == 0 for u in range(n) for v in rows[u])
    asym = sum(counts[v] > 0 and u not in sets[v] for u in range(n) for v in rows[u])
    got = stats.cpu().numpy()
    assert int(got[15]) == int(offsets[-1])
    assert (int(got[8]), int(got[9])) == (asym, dropped)  # asymmetric, dropped
