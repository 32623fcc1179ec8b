"""Batches whose cloths share the solver's tiles: what is left of a cloth after its full tiles,
and whole small cloths. Each cloth steps as a body of its own does, and an iteration of many
tiny cloths takes about as long as one of a single cloth of as many vertices (a tile for each
cloth took three times as long)."""
import ctypes as C

import numpy as np
import pytest

from licenta_amd import configs

pytestmark = pytest.mark.gpu


def _scene(n, m, k, collide):
    rng = np.random.default_rng(100 * n + m + k)
    prm = dict(configs.batched_scene(2, count=1)[0]["params"], thickness=0.004, reserved=(0, 0, 0))
    if not collide:
        prm["flags"] = configs.F_BEND_FP64
    xyz = configs.flat_grid(n, 0.01, rng, m=m) + rng.normal(0, 0.002, (n * m, 3))
    pinned = np.zeros(n * m, np.uint8)
    pinned[0] = 1
    return configs._scene(prm, xyz.astype(np.float32), configs.grid_triangles(n, m, False),
                          np.where(pinned == 1, 0.0, 1000.0).astype(np.float32), pinned,
                          configs.grid_distance_pairs_fast(n, m), name=f"c{k}")


@pytest.mark.parametrize("collide", [False, True])
@pytest.mark.parametrize("sizes", [
    [(2, 2)] * 90, [(12, 12), (3, 2)] * 9 + [(2, 64), (1 + 64, 2)], [(16, 8), (9, 9), (11, 13)] * 4,
    [(40, 33), (2, 2), (5, 5), (30, 41)]])
def test_cloths_step_as_alone(sizes, collide):
    from licenta_amd.body import ClothBody
    print(f"{len(sizes)} cloths, collide={collide}", flush=True)
    scenes = [_scene(n, m, k, collide) for k, (n, m) in enumerate(sizes)]
    batch = ClothBody.batch(scenes)
    batch.fixed_update(3)
    x, v, at = batch.positions(), batch.velocities(), 0
    for sc in scenes:
        one = ClothBody.from_scene(sc)
        one.fixed_update(3)
        n = len(sc["xyz"])
        assert np.array_equal(x[at:at + n], one.positions())
        assert np.array_equal(v[at:at + n], one.velocities())
        one.close()
        at += n
    batch.close()


def _solve_us(body):
    from licenta_amd import _abi
    ms = C.c_float()
    best = np.inf
    for _ in range(3):
        _abi.check(_abi.lib().cm_time_kernel(body.h, 0, 100, C.byref(ms)))
        best = min(best, 1e3 * ms.value)
    return best


def test_iteration_of_tiny_cloths():
    from licenta_amd.body import ClothBody
    print("8,192 cloths of 3x3", flush=True)
    us = []
    for body in (ClothBody.from_scene(_scene(272, 271, 0, False)),
                 ClothBody.batch([_scene(3, 3, k, False) for k in range(8192)])):
        us.append(_solve_us(body))
        body.close()
    assert us[1] < 2 * us[0], us


def test_iteration_of_a_small_cloth():
    """Small cloths without collisions take tiles of their size too: 16x16 took longer than
    with the solver's strips of 128 vertices, 24x24 in 5 tiles as long as 90x90 in 64."""
    from licenta_amd.body import ClothBody
    us = []
    for n, collide in ((24, False), (24, True)):
        print(f"{n}x{n}, collide={collide}", flush=True)
        body = ClothBody.from_scene(_scene(n, n, 0, collide))
        us.append(_solve_us(body))
        body.close()
    assert us[0] < 1.3 * us[1], us
