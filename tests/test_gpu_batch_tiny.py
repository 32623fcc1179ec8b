"""A batch of many tiny cloths between larger ones, whose boxes a wave collects in three ways:
each cloth steps as a body of its own does."""
import numpy as np
import pytest

from licenta_amd import configs
from test_gpu_batch import _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[(2, 2)] * 70, [(2, 2), (9, 9), (3, 2), (40, 33), (2, 3)] * 3,
                                   [(25, 30), (3, 3), (4, 3), (60, 50)]])
def test_tiny_cloths(sizes):
    from licenta_amd.body import ClothBody
    print(f"batch of {len(sizes)} cloths", flush=True)
    rng = np.random.default_rng(len(sizes))
    prm = dict(configs.batched_scene(2, count=1)[0]["params"], thickness=0.004, reserved=(0, 0, 0))
    scenes = []
    for k, (nx, ny) in enumerate(sizes):
        xyz = configs.flat_grid(nx, 0.01, rng, m=ny) + rng.normal(0, 0.003, (nx * ny, 3)) + 0.1 * k
        scenes.append(configs._scene(dict(prm), xyz.astype(np.float32),
                                     configs.grid_triangles(nx, ny, False),
                                     np.full(nx * ny, 1000.0, np.float32),
                                     np.zeros(nx * ny, np.uint8),
                                     configs.grid_distance_pairs_fast(nx, ny), name=f"c{k}"))
    singles = [ClothBody.from_scene(s) for s in scenes]
    batch = ClothBody.batch(scenes, prm)
    for _ in range(2):
        batch.fixed_update(1)
        for b in singles:
            b.fixed_update(1)
        _compare(batch, singles, scenes)
    assert batch.counts()["pairs"] > 0
    batch.close()
    for b in singles:
        b.close()
