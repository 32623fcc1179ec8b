"""The tiled Jacobi solver against the oracle at the edges of its tile shapes: fewer
vertices than a patch, one more than a tile, both workgroup sizes, the three tile sizes
of colliding cloths, a tile whose halo needs more than 64 KiB of LDS."""
import numpy as np
import pytest

from licenta_amd import configs
from test_gpu_body import run_scene

pytestmark = pytest.mark.gpu


def _grid(n, m, collide):
    rng = np.random.default_rng(100 * n + m)
    params = dict(configs.config_scene(0, 8)["params"])
    if not collide:
        params["flags"] = configs.F_BEND_FP64
    pinned = np.zeros(n * m, np.uint8)
    pinned[0] = 1
    inv_mass = np.where(pinned == 1, 0.0, 1000.0).astype(np.float32)
    return configs._scene(params, configs.flat_grid(n, 0.01, rng, m=m),
                          configs.grid_triangles(n, m, False), inv_mass, pinned,
                          configs.grid_distance_pairs_fast(n, m), name=f"grid_{n}x{m}")


@pytest.mark.parametrize("n,m,collide", [
    (2, 2, False), (2, 2, True), (16, 8, False), (3, 43, False), (11, 3, True), (65, 2, True),
    (111, 111, True), (182, 181, True)])
def test_grid_tiles(oracle_mod, n, m, collide):
    print(f"tiles of a {n}x{m} grid, collide={collide}", flush=True)
    run_scene(oracle_mod, _grid(n, m, collide), 2)


def test_fan_tile_with_large_halo(oracle_mod):
    """A fan whose centre holds 3,060 slots: a tile of one vertex with 1,531 others in
    its halo."""
    m = 1530
    ang = np.linspace(0.0, 1.9 * np.pi, m + 1)
    rim = np.stack([0.3 + 0.05 * np.cos(ang), np.full_like(ang, 0.4), 0.3 + 0.05 * np.sin(ang)], 1)
    xyz = np.vstack([[0.3, 0.4, 0.3], rim]).astype(np.float32)
    tri = np.array([[0, i, i + 1] for i in range(1, m + 1)], dtype=np.uint32)
    params = dict(configs.config_scene(0, 8)["params"])
    params["flags"] = configs.F_BEND_FP64
    sc = configs._scene(params, xyz, tri, np.full(len(xyz), 1000.0, np.float32), name="fan")
    run_scene(oracle_mod, sc, 2)
