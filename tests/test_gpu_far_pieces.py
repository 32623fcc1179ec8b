"""The pair query of scenes much larger than their triangles: a vertex far from its cloth, and
the cloths of a batch far from each other. The walk's quantised boxes must not make it pass
every node: the pairs are the exact walk's, and it takes about as long as without the distance
(it took 40 and 15 times as long; the bound is 6 times and the launches)."""
import ctypes as C

import numpy as np
import pytest

from licenta_amd import configs

pytestmark = pytest.mark.gpu


def _scene(n, seed):
    rng = np.random.default_rng(seed)
    params = dict(configs.batched_scene(2, count=1)[0]["params"], thickness=0.002)
    return configs._scene(params, configs.flat_grid(n, 0.01, rng), configs.grid_triangles(n, n, False),
                          np.full(n * n, 1000.0, np.float32), np.zeros(n * n, np.uint8),
                          configs.grid_distance_pairs_fast(n, n), name=f"sheet_{n}")


def _traverse_us(body):
    from licenta_amd import _abi
    ms = C.c_float()
    best = np.inf
    for _ in range(3):
        _abi.check(_abi.lib().cm_time_kernel(body.h, 2, 4, C.byref(ms)))
        best = min(best, 1e3 * ms.value)
    return best


@pytest.mark.parametrize("n", [64, 150])
def test_vertex_far_away(oracle_mod, n):
    from licenta_amd.body import ClothBody
    us = []
    for far in (0.0, 1e5, 1e30, np.inf):
        print(f"{n}x{n}, last vertex {far} away", flush=True)
        body = ClothBody.from_scene(_scene(n, n))
        x = body.buffer("x")[:, :3].copy()
        x[-1, 0] += np.float32(far)
        body.set_state(x, np.zeros_like(x))
        body.fixed_update(1)
        tree = [body.buffer(k) for k in ("lefts", "rights", "aabb_min", "aabb_max", "rmll", "rmlr")]
        want, _ = oracle_mod.pairs(tree[0], tree[1], tree[2][:, :3], tree[3][:, :3], *tree[4:], 64)
        assert np.array_equal(body.pairs(), want)
        us.append(_traverse_us(body))
        body.close()
    assert max(us[1:]) < 6 * us[0] + 100, us


def test_cloths_far_apart():
    from licenta_amd.body import ClothBody
    us = []
    for gap in (0.0, 1000.0):
        print(f"24 cloths {gap} apart", flush=True)
        scenes = [_scene(64, k) for k in range(24)]
        for k, sc in enumerate(scenes):
            sc["xyz"] = (sc["xyz"] + np.float32([gap * k, 0, 0])).astype(np.float32)
        body = ClothBody.batch(scenes)
        body.fixed_update(1)
        assert body.counts()["pairs"] > 0
        us.append(_traverse_us(body))
        body.close()
    assert us[1] < 6 * us[0] + 100, us
