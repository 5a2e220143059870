"""The autotuner times leaf sizes only where the search that reads them runs; a
choice among equal ones would be noise, kept for larger calls of the same key."""
import pytest

from paragram_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,leaves", [(20_000, {32}), (3 << 16, {32}), ((3 << 16) + 1, {8, 16, 32})])
def test_leaf_sizes_timed(gpu, n, leaves):
    import torch

    from paragram_amd import autotune

    print(f"autotune: leaf sizes timed at {n} points", flush=True)
    cfg = autotune.tune(torch.from_numpy(workloads.uniform(n, 6)).to(gpu), force=True)
    assert {int(k.split("/")[0]) for k in cfg["ms"]} == leaves
    assert cfg["leaf_size"] in leaves and cfg["preclip"] in autotune.PRECLIPS
