"""The lane walk on either side of the leaf counts where its stack and candidate rows change:
lists longer than the candidate rows, and stacks deeper than the rows of the stack."""
import numpy as np
import pytest

from test_gpu_quant_walk import _gpu_pairs, _keys, _tree

pytestmark = pytest.mark.gpu


def _sheet(oracle_mod, t, size):
    """Boxes in the order of their Morton codes, as a scene's tree has them."""
    rng = np.random.default_rng(t)
    lo = rng.uniform(0, 1, (t, 3)).astype(np.float32)
    lo[:, 1] *= 0.01
    keys = np.array(oracle_mod.morton63(lo), np.uint64)
    order = np.argsort(keys, kind="stable")
    left, right, _, _ = oracle_mod.build(keys[order], True, np.zeros(2 * t - 1, np.int32))
    mn, mx = np.zeros((2 * t - 1, 3), np.float32), np.zeros((2 * t - 1, 3), np.float32)
    mn[t - 1:] = lo[order]
    mx[t - 1:] = mn[t - 1:] + rng.uniform(0, size / np.sqrt(t), (t, 3)).astype(np.float32)
    return (left, right) + oracle_mod.refit(left, right, mn, mx)


@pytest.mark.parametrize("t,size,cap", [(131072, 8.0, 64), (131073, 8.0, 64), (262144, 8.0, 48),
                                        (262145, 8.0, 48), (327680, 7.0, 40), (327681, 7.0, 40)])
def test_rows(oracle_mod, t, size, cap):
    print(f"walk t={t} size={size} cap={cap}", flush=True)
    tree = _sheet(oracle_mod, t, size)
    want, warn = oracle_mod.pairs(*tree, cap)
    assert len(want) > 16 * t and warn
    got, gwarn = _gpu_pairs(*tree, cap)
    assert np.array_equal(got, want)
    assert gwarn == warn


@pytest.mark.parametrize("t", [140000, 270000, 330000])
def test_deep_stacks(oracle_mod, t):
    print(f"deep walk t={t}", flush=True)
    tree = _tree(oracle_mod, _keys("deep", t), 2.0, t)
    want, warn = oracle_mod.pairs(*tree, 16)
    got, gwarn = _gpu_pairs(*tree, 16)
    assert np.array_equal(got, want)
    assert gwarn == warn
