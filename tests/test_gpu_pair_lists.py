"""The pair list's compaction where its route changes: tiles that add up the sums before
theirs up to 1,024 tiles of 128 leaves, a scan beyond; leaves without pairs, a last tile of
one leaf, several workgroups a tile; and the Morton keys' box by one workgroup or by all."""
import numpy as np
import pytest

from test_gpu_lbvh import check, dev, f4, lib, stream, vp
from test_gpu_quant_walk import _gpu_pairs, _keys

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _line(oracle_mod, t, near):
    """Boxes along a line, each meeting up to `near` of its neighbours on either side."""
    rng = np.random.default_rng(t)
    left, right, _, _ = oracle_mod.build(_keys("unique", t), True, np.zeros(2 * t - 1, np.int32))
    mn, mx = np.zeros((2 * t - 1, 3), np.float32), np.zeros((2 * t - 1, 3), np.float32)
    mn[t - 1:, 0] = np.arange(t)
    mx[t - 1:] = mn[t - 1:] + rng.uniform(0, near, (t, 1)).astype(np.float32)
    return (left, right) + oracle_mod.refit(left, right, mn, mx)


@pytest.mark.parametrize("t,near,cap", [(129, 0, 8), (257, 200, 64), (40000, 60, 100),
                                        (131072, 12, 24), (131073, 40, 24)])
def test_pair_list(oracle_mod, t, near, cap):
    print(f"pair list t={t} cap={cap}", flush=True)
    tree = _line(oracle_mod, t, near)
    want, warn = oracle_mod.pairs(*tree, cap)
    got, gwarn = _gpu_pairs(*tree, cap)
    assert np.array_equal(got, want)
    assert gwarn == warn


@pytest.mark.parametrize("t", [1, 256, 131072, 131073])
def test_keys_of_box(oracle_mod, t):
    rng = np.random.default_rng(t)
    x = rng.uniform(-3, 5, (t + 2, 3)).astype(np.float32)
    tri = np.zeros((t, 4), np.int32)
    tri[:, :3] = np.arange(t)[:, None] + np.arange(3)
    dmin = torch.zeros((2 * t - 1, 4), dtype=torch.float32, device="cuda")
    dmax = torch.zeros((2 * t - 1, 4), dtype=torch.float32, device="cuda")
    dk = torch.zeros(t, dtype=torch.int64, device="cuda")
    dx, dt = dev(f4(x)), dev(tri)
    check(lib().cm_tri_update(t + 2, t, vp(dx), vp(dx), vp(dt), 0.003, 30, 1, vp(dmin), vp(dmax),
                              vp(dk), stream()))
    torch.cuda.synchronize()
    th = np.float32(0.003)
    p = x[tri[:, :3]]
    mn, mx = (p - th).min(1), (p + th).max(1)
    cen = (mn + (mx - mn) / np.float32(2)).astype(np.float32)
    want = oracle_mod.morton30(cen, cen.min(0), cen.max(0))
    assert np.array_equal(dk.cpu().numpy().view(np.uint64), want)
