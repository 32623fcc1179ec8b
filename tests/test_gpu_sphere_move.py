"""A sphere moved between substeps without a wait: each substep sees the sphere that was set
before it, as a body created with that sphere does."""
import numpy as np
import pytest

from licenta_amd import configs

pytestmark = pytest.mark.gpu


def _scene(n, centre, radius, with_sphere):
    rng = np.random.default_rng(3)
    params = dict(configs.config_scene(0, 8)["params"], thickness=0.002)
    params["flags"] = configs.F_BEND_FP64 | (configs.F_SPHERE if with_sphere else 0)
    params.update(sphere_center=centre, sphere_radius=radius)
    return configs._scene(params, configs.flat_grid(n, 0.01, rng), configs.grid_triangles(n, n, False),
                          np.full(n * n, 1000.0, np.float32), None,
                          configs.grid_distance_pairs_fast(n, n), name=f"sphere_{n}")


@pytest.mark.parametrize("n,first", [(2, True), (17, True), (33, False)])
def test_moved_sphere(n, first):
    from licenta_amd.body import ClothBody
    print(f"moved sphere {n}x{n}", flush=True)
    sc = _scene(n, (0.0, -1.0, 0.0), 0.1, first)
    xyz = sc["xyz"]
    v = np.full_like(xyz, 0.0)
    v[:, 1] = -1.0
    body = ClothBody.from_scene(sc)
    body.set_state(xyz, v)
    mid = xyz.mean(0)
    path = [tuple(float(c) for c in mid - np.array([0.01 * k, 0.13 + 0.005 * k, 0.0]))
            for k in range(5)]
    for c in path:  # no read and no wait in between
        body.set_sphere_pos(c, 0.12)
        body.fixed_update(1)
    x, vel = xyz, v
    moved = False
    for c in path:
        one = ClothBody.from_scene(_scene(n, c, 0.12, True))
        free = ClothBody.from_scene(_scene(n, (0.0, -9.0, 0.0), 0.1, False))
        for b in (one, free):
            b.set_state(x, vel)
            b.fixed_update(1)
        x, vel = one.positions(), one.velocities()
        moved |= not np.array_equal(x, free.positions())
        one.close()
        free.close()
    assert np.array_equal(body.positions(), x)
    assert np.array_equal(body.velocities(), vel)
    assert moved or n == 2
    body.close()
