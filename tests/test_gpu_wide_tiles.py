"""A vertex in more than a thousand bends that share no other vertex: with their positions its
tile does not fit the LDS and reads them from memory. Such a mesh steps as the oracle does and
is differentiable (the layout was refused to the adjoint), alone and beside a cloth of many
tiles."""
import numpy as np
import pytest

from licenta_amd import configs
from test_gpu_adjoint import TOL, _gpu_grads, _oracle_grads, scaled_err
from test_gpu_body import run_scene

pytestmark = pytest.mark.gpu


def _flaps(count, sheet):
    """`count` flaps of two triangles about vertex 0: (0, a, b) and (b, a, d)."""
    rng = np.random.default_rng(count)
    a = rng.normal(0, 1, (count, 3))
    a *= 0.05 / np.linalg.norm(a, axis=1, keepdims=True)
    side = np.cross(a, rng.normal(0, 1, (count, 3)))
    side *= 0.02 / np.linalg.norm(side, axis=1, keepdims=True)
    out = np.cross(side, a)
    out *= 0.015 / np.linalg.norm(out, axis=1, keepdims=True)
    tips = np.stack([a - side, a + side, 1.4 * a + out], 1).reshape(-1, 3)
    xyz = np.vstack([np.zeros((1, 3)), tips]) + 0.5
    i = 1 + 3 * np.arange(count)
    tri = np.stack([0 * i, i, i + 1, i + 1, i, i + 2], 1).reshape(-1, 3)
    pairs = np.stack([i, i + 1, i, i + 2, i + 1, i + 2], 1).reshape(-1, 2)
    if sheet:
        at = len(xyz)
        xyz = np.vstack([xyz, configs.flat_grid(sheet, 0.01, rng) + rng.normal(0, 0.002, (sheet * sheet, 3))])
        tri = np.vstack([tri, configs.grid_triangles(sheet, sheet, False).astype(np.int64) + at])
        pairs = np.vstack([pairs, configs.grid_distance_pairs_fast(sheet, sheet) + at])
    params = dict(configs.config_scene(3, 8)["params"], flags=configs.F_BEND_FP64, timestep=1.0 / 240.0)
    return configs._scene(params, xyz.astype(np.float32), tri.astype(np.uint32),
                          np.full(len(xyz), 1000.0, np.float32), None, pairs.astype(np.int32),
                          name=f"flaps_{count}_{sheet}")


@pytest.mark.parametrize("count,sheet", [(1400, 0), (3000, 0), (1400, 80), (600, 80)])
def test_flaps(oracle_mod, count, sheet):
    from licenta_amd.body import ClothBody
    print(f"{count} flaps, sheet of {sheet}^2", flush=True)
    sc = _flaps(count, sheet)
    run_scene(oracle_mod, sc, 2, check_tree=False)
    body = ClothBody.from_scene(sc)
    c = body.counts()
    assert c["b"] >= count
    rng = np.random.default_rng(3)
    kd = rng.uniform(0.3, 0.95, c["s"]).astype(np.float32)
    kb = rng.uniform(0.05, 0.3, c["b"]).astype(np.float32)
    v0 = rng.normal(0.0, 0.05, (c["n"], 3)).astype(np.float32)
    target = sc["xyz"].astype(np.float64) + rng.normal(0.0, 0.01, (c["n"], 3))
    body.set_stiffness(kd, kb)
    body.set_state(sc["xyz"], v0)
    ref, _, _ = _oracle_grads(oracle_mod, sc, body, kd, kb, v0, target, 2)
    g, _ = _gpu_grads(body, target, 2, 1)
    body.close()
    for k in ("kd", "kb", "x", "v"):
        assert np.abs(ref[k]).max() > 0
        assert scaled_err(g[k], ref[k]) <= TOL, (k, scaled_err(g[k], ref[k]))
