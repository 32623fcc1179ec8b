"""A body whose candidate capacities add up to more than 2^31: the same contacts as with
small capacities. (At the default capacities this is a body of 6.7 M triangles and more.)"""
import numpy as np
import pytest

from test_gpu_narrow_tiles import _scene

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_candidate_capacity_above_2_31():
    from licenta_amd.body import ClothBody
    if torch.cuda.mem_get_info()[0] < 160 << 30:
        pytest.skip("needs 110 GB of device memory")
    sc, v = _scene(79, 79, 0.003, 0.004)
    t = len(sc["tri"])
    got = []
    for vf, ee in ((0, 0), (6 * t, 9 * t)):
        print(f"candidate capacities {vf} and {ee} a triangle", flush=True)
        # the candidates are also bounded by 6 and 9 for each pair that fits: t a triangle
        sc["params"] = dict(sc["params"], pair_cap=t, reserved=(vf, ee, 0))
        assert vf == 0 or (vf + ee) * t > 1 << 31
        body = ClothBody.from_scene(sc)
        body.set_state(sc["xyz"], v)
        for _ in range(2):
            body.fixed_update(1)
        got.append((body.counts(), body.pairs(), *body.contacts(), body.positions()))
        body.close()
    assert got[0][0]["vf"] > 0 and got[0][0]["ee"] > 0
    assert got[0][0] == got[1][0]
    for a, b in zip(got[0][1:], got[1][1:]):
        assert np.array_equal(a, b)
