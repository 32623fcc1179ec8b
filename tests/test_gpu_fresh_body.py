"""Kernels timed on a body that has not stepped: a batch has no cloth roots before its first
build, so the traversal finds nothing to walk, and the steps that follow are those of a body
that was not timed."""
import ctypes as C

import numpy as np
import pytest

from licenta_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cloths", [0, 4, 24])  # one body; a batch walked by groups, by lanes
def test_timed_before_a_step(cloths):
    from licenta_amd import _abi
    from licenta_amd.body import ClothBody
    print(f"{cloths} cloths of 64x64", flush=True)
    scenes = configs.batched_scene(4, count=max(cloths, 1))

    def make():
        return ClothBody.batch(scenes) if cloths else ClothBody.from_scene(scenes[0])

    timed, plain = make(), make()
    for which in (2, 3):  # traversal, CCD plan
        ms = C.c_float()
        _abi.check(_abi.lib().cm_time_kernel(timed.h, which, 2, C.byref(ms)))
    assert timed.counts()["pairs"] == 0
    for body in (timed, plain):
        body.fixed_update(2)
    assert plain.counts()["pairs"] > 0
    assert np.array_equal(timed.positions(), plain.positions())
    assert np.array_equal(timed.pairs(), plain.pairs())
    timed.close()
    plain.close()
