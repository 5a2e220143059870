"""The statistics count every cell once, also the cells that tier 0 gives up on:
at its tests (scans, grids with exact ties), on capacity (a hub) and inside a
predicted cube that cut them."""
import numpy as np
import pytest

from paragram_amd import workloads

pytestmark = pytest.mark.gpu


def grid():
    return (np.unique(np.random.default_rng(1).integers(0, 16, (4000, 3)), axis=0) / 16.0).astype(np.float32)


def hub():
    r = np.random.default_rng(3)
    d = r.standard_normal((200, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return np.concatenate([np.zeros((1, 3)), d, r.random((1500, 3)) * 2.0 + 2.0]).astype(np.float32)


INPUTS = {
    "scan": lambda: workloads.lidar_batch(3, max_clouds=1)[0][:30_000],
    "small_grid": grid,
    "hub": hub,
    "uniform": lambda: workloads.uniform(10_001, 4),
}


@pytest.mark.parametrize("cube", [False, True])
@pytest.mark.parametrize("name", list(INPUTS))
def test_every_cell_is_counted_once(gpu, name, cube):
    import torch

    from paragram_amd import _engine
    from paragram_amd._backend import _C

    print(f"cell count: {name}, predicted cube {cube}", flush=True)
    pts = torch.from_numpy(np.ascontiguousarray(INPUTS[name](), np.float32)).to(gpu)
    n = pts.shape[0]
    h = torch.full((n,), 1e-3, device=gpu) if cube else None  # (cuts nearly every cell)
    ins = _engine.Instrument()
    _engine.build_diagram(_C.lib, pts, None, instrument=ins, init_h=h)
    print({k: ins.stats[k] for k in ("cells", "bail_test", "bail_vertex", "promoted")}, flush=True)
    assert ins.stats["cells"] == n
    if name in ("scan", "small_grid") and not cube:  # (a cube that cuts ends a cell before its tests)
        assert ins.stats["bail_test"] > 0


def test_every_cell_of_a_batch_is_counted_once(gpu):
    import torch

    from paragram_amd import _engine
    from paragram_amd._backend import _C

    parts = [INPUTS["scan"]()[:9000], grid(), np.zeros((0, 3), np.float32), hub(), workloads.uniform(1, 1)]
    pts = torch.from_numpy(np.concatenate(parts).astype(np.float32)).to(gpu)
    offsets = np.concatenate([[0], np.cumsum([p.shape[0] for p in parts])])
    ins = _engine.Instrument()
    _engine.build_diagram(_C.lib, pts, None, instrument=ins, clouds=offsets)
    assert ins.stats["cells"] == pts.shape[0] and ins.stats["bail_test"] > 0
