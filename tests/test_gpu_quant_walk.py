"""The tree walk through quantised node boxes against the oracle's exact walk: small and
odd trees, tied codes (nodes with two parents), trees deep enough to fill the 63-entry
stack, scenes without extent along an axis, and trees the quantised walk must leave to
the exact one (NaN and infinite boxes, boxes that do not hold what lies below, renumbered
nodes)."""
import numpy as np
import pytest

from test_gpu_lbvh import check, dev, f4, lib, stream, vp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _gpu_pairs(left, right, mn, mx, rl, rr, cap):
    t = len(left) + 1
    L = lib()
    nb = L.cm_lbvh_pairs_temp_bytes(t, cap)
    tmp = torch.empty(nb, dtype=torch.uint8, device="cuda")
    out = torch.zeros(2 * t * cap, dtype=torch.int32, device="cuda")
    cnt = torch.zeros(1, dtype=torch.int32, device="cuda")
    warn = torch.zeros(1, dtype=torch.int32, device="cuda")
    a = [dev(x) for x in (left, right, f4(mn), f4(mx), rl, rr)]
    check(L.cm_lbvh_pairs(t, *[vp(x) for x in a], cap, vp(out), vp(cnt), vp(warn), vp(tmp), nb,
                          stream()))
    torch.cuda.synchronize()
    n = int(cnt.cpu()[0])
    return out.cpu().numpy()[:2 * n].reshape(-1, 2), int(warn.cpu()[0]) & 0xFFFF


def _tree(oracle_mod, keys, size, seed, flat=False):
    rng = np.random.default_rng(seed)
    t = len(keys)
    left, right, _, _ = oracle_mod.build(keys, True, np.zeros(2 * t - 1, np.int32))
    lo = rng.uniform(0, 1, (t, 3)).astype(np.float32)
    mn, mx = np.zeros((2 * t - 1, 3), np.float32), np.zeros((2 * t - 1, 3), np.float32)
    mn[t - 1:], mx[t - 1:] = lo, lo + rng.uniform(0, size, (t, 3)).astype(np.float32)
    if flat:  # no extent along y, a tiny one far from the origin along z
        mn[t - 1:, 1] = mx[t - 1:, 1] = 0.25
        mn[t - 1:, 2], mx[t - 1:, 2] = 1e6 + mn[t - 1:, 2], 1e6 + mx[t - 1:, 2]
    return (left, right) + oracle_mod.refit(left, right, mn, mx)


def _keys(kind, t):
    rng = np.random.default_rng(t)
    if kind == "unique":
        return np.unique(rng.integers(0, 1 << 62, 2 * t, dtype=np.int64))[:t].astype(np.uint64)
    if kind == "ties":
        return np.sort(rng.integers(0, max(2, t // 50), t).astype(np.uint64) << np.uint64(20))
    # two leaves a bit length, then equal codes: 62 nested levels and 12 more
    k = [1 << b for b in range(1, 62)] + [(1 << b) + 1 for b in range(1, 62)] + [0] * t
    return np.sort(np.array(k, np.uint64))


@pytest.mark.parametrize("kind,t,size,cap", [
    ("unique", 2, 0.5, 4), ("unique", 3, 0.9, 1), ("unique", 4, 0.9, 8), ("unique", 7, 0.9, 8),
    ("unique", 129, 0.4, 16), ("unique", 5000, 0.05, 64), ("unique", 5000, 0.3, 3),
    ("ties", 257, 0.3, 32), ("ties", 20000, 0.03, 64), ("deep", 1, 2.0, 200),
    ("deep", 4096, 2.0, 16)])
def test_walk_matches_oracle(oracle_mod, kind, t, size, cap):
    print(f"walk {kind} t={t} size={size} cap={cap}", flush=True)
    tree = _tree(oracle_mod, _keys(kind, t), size, t)
    want, warn = oracle_mod.pairs(*tree, cap)
    got, gwarn = _gpu_pairs(*tree, cap)
    assert np.array_equal(got, want)
    assert gwarn == warn


def test_flat_scene(oracle_mod):
    tree = _tree(oracle_mod, _keys("unique", 2000), 0.05, 3, flat=True)
    want, warn = oracle_mod.pairs(*tree, 64)
    got, gwarn = _gpu_pairs(*tree, 64)
    assert np.array_equal(got, want)
    assert gwarn == warn


@pytest.mark.parametrize("what", ["nan", "inf", "loose", "renumbered"])
def test_irregular_trees(oracle_mod, what):
    print(f"irregular tree: {what}", flush=True)
    t = 3000
    left, right, mn, mx, rl, rr = [np.array(a) for a in
                                   _tree(oracle_mod, _keys("ties", t), 0.1, 5)]
    rng = np.random.default_rng(9)
    if what in ("nan", "inf"):
        for k in rng.integers(0, t, 20):
            (mn if k % 2 else mx)[t - 1 + k, k % 3] = np.nan if what == "nan" else np.inf
        mn, mx, rl, rr = [np.array(a) for a in oracle_mod.refit(left, right, mn, mx)]
    elif what == "loose":
        k = rng.integers(1, t - 1, 200)
        mx[k] -= 0.05
    else:  # the root stays node 0
        new = np.concatenate([[0], 1 + rng.permutation(t - 2)])
        at = np.concatenate([new, np.arange(t - 1, 2 * t - 1)])
        l2, r2, rl2, rr2 = (np.empty_like(left) for _ in range(4))
        l2[new], r2[new], rl2[new], rr2[new] = at[left], at[right], rl, rr
        m2, x2 = np.empty_like(mn), np.empty_like(mx)
        m2[at], x2[at] = mn, mx
        left, right, mn, mx, rl, rr = l2, r2, m2, x2, rl2, rr2
    want, warn = oracle_mod.pairs(left, right, mn, mx, rl, rr, 32)
    got, gwarn = _gpu_pairs(left, right, mn, mx, rl, rr, 32)
    assert np.array_equal(got, want)
    assert gwarn == warn
