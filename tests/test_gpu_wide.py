"""The 16-wide form of the hierarchy against the CPU oracle, bit for bit, where
it can go wrong: cloud sizes at the edges of its classes (32 * 8^k points), leaf
sizes up to a whole class, a chain of clusters whose nodes have more than 16
children (walked as binary nodes), cells of many faces (built by the larger
tiers, a wave per cell), and batches whose clouds lie in different classes.  Whole-number outputs: no tolerance."""
import numpy as np
import pytest

from paragram_amd import workloads
from tests.test_gpu_batch import assert_same, batch, single
from tests.test_gpu_parity import assert_matches_oracle, run

pytestmark = pytest.mark.gpu


def chain(per_cluster: int, rest: int) -> np.ndarray:
    """30 clusters, each leaving the subtree at the next bit of the Morton key,
    and ``rest`` points in the corner cell: the largest subtree of every split
    is the rest of the chain."""
    rng = np.random.default_rng(31)
    parts = [np.ones((1, 3))]
    for level in range(30):
        axis, j = level % 3, level // 3 + 1
        c = rng.random((per_cluster, 3)) * 2.0 ** -(j + 1)
        c[:, axis] += 2.0**-j
        c[:, (axis + 1) % 3] *= 1.0 if axis < 2 else 0.5
        parts.append(c)
    parts.append(rng.random((rest, 3)) * 2.0**-11)
    return np.concatenate(parts).astype(np.float32)


@pytest.mark.parametrize("n", [31, 32, 33, 34, 255, 256, 257, 2047, 2048, 2049])
@pytest.mark.parametrize("leaf", [8, 32])
def test_class_edges(gpu, n, leaf):
    print(f"wide form: n={n} leaf_size={leaf}", flush=True)
    pts = workloads.uniform(n, 700 + n)
    assert_matches_oracle(run(gpu, pts, leaf_size=leaf), pts)


@pytest.mark.parametrize("n", [3, 5, 4095, 4096, 4097, 6143, 6144, 6145])
def test_cells_per_wave_edges(gpu, n):
    """Sizes at which a wave takes one, two or four cells (2048 is among the above)."""
    print(f"cells per wave: n={n}", flush=True)
    pts = workloads.uniform(n, 300 + n)
    assert_matches_oracle(run(gpu, pts), pts)


@pytest.mark.parametrize("per_cluster,rest", [(20, 300), (1, 40), (70, 2100)])
def test_more_than_16_children(gpu, per_cluster, rest):
    pts = chain(per_cluster, rest)
    print(f"wide form: chain of {pts.shape[0]} points", flush=True)
    assert_matches_oracle(run(gpu, pts), pts)
    w = np.random.default_rng(5).uniform(0, 1e-7, pts.shape[0]).astype(np.float32)
    assert_matches_oracle(run(gpu, pts, w), pts, w)


@pytest.mark.parametrize("faces", [40, 97, 98, 99, 130, 257, 258, 259, 500])
def test_hub_cells(gpu, faces):
    """A point amid ``faces`` points of a sphere: its cell has that many faces and
    about twice the vertices, at the edges of the larger tiers' capacities."""
    print(f"wide form: hub of {faces} faces", flush=True)
    rng = np.random.default_rng(faces)
    d = rng.standard_normal((faces, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    far = rng.random((1500, 3)) * 2.0 + 2.0
    pts = np.concatenate([np.zeros((1, 3)), d, far]).astype(np.float32)
    assert_matches_oracle(run(gpu, pts), pts)


def test_batch_of_classes(gpu):
    sizes = [33, 1, 2049, 32, 257, 0, 40, 256, 2, 300]
    print(f"wide form: batch of {sizes}", flush=True)
    rng = np.random.default_rng(8)
    clouds = [rng.random((m, 3)).astype(np.float32) for m in sizes] + [chain(20, 300)]
    for k, got in enumerate(batch(gpu, clouds)):
        if clouds[k].shape[0]:
            assert_same(got, single(gpu, clouds[k]), f"cloud {k} ({clouds[k].shape[0]} points)")
