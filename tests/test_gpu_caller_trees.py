"""cm_lbvh_pairs on trees that no build of the library makes: children side by side and
boxes that hold what lies below, as the quantised walk takes them, but leaves in any order
and nodes with several parents or none. The oracle's walk gives the pairs."""
import numpy as np
import pytest

from test_gpu_quant_walk import _gpu_pairs, _keys, _tree
from test_gpu_walk_shapes import _sheet

pytestmark = pytest.mark.gpu


def _refit(oracle_mod, left, right, lo, hi):
    t = len(left) + 1
    left, right = np.array(left, np.int32), np.array(right, np.int32)
    mn, mx = np.zeros((2 * t - 1, 3), np.float32), np.zeros((2 * t - 1, 3), np.float32)
    mn[t - 1:], mx[t - 1:] = lo, hi
    return (left, right) + oracle_mod.refit(left, right, mn, mx)


def _check(oracle_mod, tree, cap):
    want, warn = oracle_mod.pairs(*tree, cap)
    got, gwarn = _gpu_pairs(*tree, cap)
    assert np.array_equal(got, want)
    assert gwarn == warn


@pytest.mark.parametrize("cap", [1, 8, 79, 80])
def test_leaf_right_of_its_right_neighbour(oracle_mod, cap):
    """Node 0 = (node 1, leaf 2), node 1 = (node 2, leaf 3), node 2 = (leaf 0, leaf 1): the
    left subtree's rightmost leaf lies beyond the right leaf."""
    print(f"leaf order, cap {cap}", flush=True)
    tree = _refit(oracle_mod, [1, 2, 3], [5, 6, 4], np.zeros((4, 3)), np.ones((4, 3)))
    _check(oracle_mod, tree, cap)


def _random_tree(oracle_mod, rng):
    """Up to 8 leaves; a child is the leaf or the later node of its number."""
    t = int(rng.integers(2, 9))
    left, right = [], []
    for i in range(t - 1):
        sp = int(rng.integers(0, t - 1))
        kids = [c if i < c < t - 1 and rng.integers(0, 2) else t - 1 + c for c in (sp, sp + 1)]
        left.append(kids[0])
        right.append(kids[1])
    lo = rng.uniform(0, 1, (t, 3))
    return _refit(oracle_mod, left, right, lo, lo + rng.uniform(0, 1.5, (t, 3)))


@pytest.mark.parametrize("cap", [2, 16, 80])
def test_random_small_trees(oracle_mod, cap):
    rng = np.random.default_rng(cap)
    for k in range(60):
        print(f"random tree {k}, cap {cap}", flush=True)
        _check(oracle_mod, _random_tree(oracle_mod, rng), cap)


def _shared(oracle_mod, levels, chain):
    """`levels` pairs of nodes, each node of a pair above both of the next, then a chain: the
    chain is walked once for each of the 2^levels paths to it. The leaves of low numbers lie
    in no node, between the chain's leaves, which the last but one of them meets."""
    b = 2 * levels + 1
    t = b + chain + 1
    left, right = list(range(1, t)), list(range(2, t + 1))
    for k in range(1, levels):  # nodes 2k - 1 and 2k have the children 2k + 1 and 2k + 2
        left[2 * k - 1], right[2 * k - 1] = 2 * k + 1, 2 * k + 2
        left[2 * k], right[2 * k] = 2 * k + 1, 2 * k + 2
    for i in range(b - 2, t - 1):  # leaf s, then node s + 1
        s = max(i, b - 1)
        left[i], right[i] = t - 1 + s, s + 1
    right[t - 2] = 2 * t - 2
    lo = np.zeros((t, 3))
    lo[:b - 1, 0] = 5.0
    lo[b - 2, 0] = 0.5
    lo[t - 1, 0] = 10.0
    return _refit(oracle_mod, left, right, lo, lo + 1.0)


@pytest.mark.parametrize("levels,chain,cap", [(8, 24, 16), (8, 25, 16), (8, 40, 79), (11, 38, 79),
                                              (11, 38, 80)])
def test_visit_limit(oracle_mod, levels, chain, cap):
    """Trees whose shared nodes make fewer visits than the limit, a few more and many more."""
    print(f"visit limit: {levels} levels, chain {chain}, cap {cap}", flush=True)
    tree = _shared(oracle_mod, levels, chain)
    want, warn = oracle_mod.pairs(*tree, cap)
    limited = (2 << levels) - 1 + (chain << levels) > 64 * (len(tree[0]) + 1) + 4096
    assert bool(warn & 2) == limited
    _check(oracle_mod, tree, cap)


@pytest.mark.parametrize("t,cap", [(4, 2), (4, 80), (300, 16), (300, 90), (40000, 8)])
def test_unheld_leaf_with_nan_box(oracle_mod, t, cap):
    """Leaf 0 belongs to no node (its parent holds leaves 1 and 2) and its box is NaN, which
    overlaps every box: its pairs are the leaves of the tree up to the cap."""
    print(f"NaN leaf beside a tree of {t} leaves, cap {cap}", flush=True)
    left, right, mn, mx, _, _ = _tree(oracle_mod, _keys("unique", t), 0.05, t)
    lo, hi = np.array(mn[t - 1:]), np.array(mx[t - 1:])
    lo[0] = hi[0] = np.nan
    left, right = np.array(left), np.array(right)
    parent = np.flatnonzero(left == t - 1)[0]
    left[parent], right[parent] = t, t + 1
    tree = _refit(oracle_mod, left, right, lo, hi)
    want, _ = oracle_mod.pairs(*tree, cap)
    assert (want[:, 0] == 0).sum() >= min(cap, t - 1)
    _check(oracle_mod, tree, cap)


@pytest.mark.parametrize("t,cap", [(32768, 16), (32769, 16), (32769, 100), (150001, 24)])
def test_renumbered_nodes(oracle_mod, t, cap):
    """The build's tree with its nodes in another order (the root stays node 0), up to the
    leaves from which on the exact walk takes records of its own; lists cut at the cap."""
    print(f"renumbered tree of {t} leaves, cap {cap}", flush=True)
    left, right, mn, mx, rl, rr = _sheet(oracle_mod, t, 4.0 if cap > 24 else 8.0)
    rng = np.random.default_rng(t)
    new = np.concatenate([[0], 1 + rng.permutation(t - 2)])
    at = np.concatenate([new, np.arange(t - 1, 2 * t - 1)])
    tree = [np.empty_like(a) for a in (left, right, mn, mx, rl, rr)]
    tree[0][new], tree[1][new], tree[4][new], tree[5][new] = at[left], at[right], rl, rr
    tree[2][at], tree[3][at] = mn, mx
    _check(oracle_mod, tree, cap)
