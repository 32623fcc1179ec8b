"""cm_autotune on bodies whose traversal has no chunks and no budget: it tunes the tile size and
leaves the other two as they are, instead of reporting whichever of equal runs was shorter."""
import numpy as np
import pytest

from licenta_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cap,groups", [(40, 64, True), (40, 79, True), (40, 80, False),
                                          (128, 64, True), (130, 64, False)])
def test_small_bodies(n, cap, groups):
    from licenta_amd.body import ClothBody
    print(f"autotune {n}x{n}, cap {cap}", flush=True)
    sc = configs.config_scene(0, n)
    sc["params"] = dict(sc["params"], pair_cap=cap)
    a, b = ClothBody.from_scene(sc), ClothBody.from_scene(sc)
    picks = b.autotune(1)
    if groups:
        assert picks["traversal_chunk"] == 4 and picks["traversal_budget"] == 0
    else:
        assert picks["traversal_budget"] in (128, 160, 200, 240)
    assert picks["tile_vertices"] in (32, 64, 128, 256)
    a.fixed_update(3)
    b.fixed_update(3)
    assert np.array_equal(a.positions(), b.positions())
    assert np.array_equal(a.pairs(), b.pairs())
    a.close()
    b.close()
