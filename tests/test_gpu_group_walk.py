"""The walk by groups of lanes where it begins and ends: its largest tree and one leaf more,
its largest cap and one more (then one lane per leaf walks), caps that make it drop hits
while it walks, trees whose leaves it leaves to the exact walk."""
import numpy as np
import pytest

from test_gpu_quant_walk import _gpu_pairs, _keys, _tree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,t,size,cap", [
    ("unique", 32768, 0.02, 16), ("unique", 32769, 0.02, 16), ("unique", 2000, 0.6, 79),
    ("unique", 2000, 0.6, 80), ("unique", 1500, 1.0, 1), ("unique", 1500, 1.0, 33),
    ("ties", 3000, 0.2, 79), ("ties", 3000, 0.2, 96), ("deep", 300, 1.5, 79),
    ("deep", 300, 1.5, 80), ("unique", 2, 0.5, 80), ("unique", 5, 1.0, 80)])
def test_walk_matches_oracle(oracle_mod, kind, t, size, cap):
    print(f"walk {kind} t={t} size={size} cap={cap}", flush=True)
    tree = _tree(oracle_mod, _keys(kind, t), size, 3 * t + cap)
    want, warn = oracle_mod.pairs(*tree, cap)
    got, gwarn = _gpu_pairs(*tree, cap)
    assert np.array_equal(got, want)
    assert gwarn == warn
