"""The radix sort where its route changes: one workgroup up to 8,192 keys, tiles that add up
each other's digit counts up to 131,072, a scan beyond; and the contact lists' sort with
more than one tile a workgroup."""
import numpy as np
import pytest

from licenta_amd import configs
from test_gpu_lbvh import run_sort

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [3, 63, 64, 65, 1023, 1025, 8191, 8192, 8193, 131072, 131073])
@pytest.mark.parametrize("bits", [8, 30, 32, 33, 63, 64])
def test_sort_routes(oracle_mod, t, bits):
    print(f"sort t={t} bits={bits}", flush=True)
    rng = np.random.default_rng(7 * t + bits)
    keys = rng.integers(0, 1 << bits, size=t, dtype=np.uint64, endpoint=False) if bits < 64 else \
        rng.integers(0, 1 << 63, size=t, dtype=np.uint64) * np.uint64(2) + np.uint64(1)
    keys[: t // 3] = keys[-1]
    rng.shuffle(keys)
    vals = rng.integers(0, 1 << 32, size=t, dtype=np.uint64).astype(np.uint32)
    gk, gv = run_sort(keys, vals, bits)
    ok, ov = oracle_mod.stable_sort(keys, vals)
    assert np.array_equal(gk, ok)
    assert np.array_equal(gv, ov)


@pytest.mark.parametrize("t", [3000, 9000, 140000])
def test_sort_carries_upper_bits(t):
    """Keys sorted by their low 32 bits keep what is above them."""
    rng = np.random.default_rng(t)
    keys = rng.integers(0, 1 << 63, size=t, dtype=np.uint64)
    keys[: t // 2] &= np.uint64(0xFFFFFFFF00000FFF)  # many equal low words
    vals = np.arange(t, dtype=np.uint32)
    gk, gv = run_sort(keys, vals, 32)
    order = np.argsort(keys & np.uint64(0xFFFFFFFF), kind="stable")
    assert np.array_equal(gk, keys[order])
    assert np.array_equal(gv, vals[order])


@pytest.mark.parametrize("n,m,tiles", [(20, 31, 1), (190, 150, 64), (420, 400, 257)])
def test_contact_lists(monkeypatch, n, m, tiles):
    """The sorted contact lists against the counted ones, with at least `tiles` tiles of
    2,048 records: the same positions bit for bit."""
    from licenta_amd.body import ClothBody
    from test_gpu_narrow_tiles import _scene
    print(f"contact lists {n}x{m}", flush=True)
    sc, v = _scene(n, m, 0.003, 0.006)
    out = []
    for mode in ("1", "0"):
        monkeypatch.setenv("CLOTHMI_SORT_CSR", mode)
        body = ClothBody.from_scene(sc)
        body.set_state(sc["xyz"], v)
        body.fixed_update(2)
        c = body.counts()
        out.append((body.positions(), body.velocities(), c["vf"] + c["ee"]))
        body.close()
    assert out[0][2] == out[1][2] and -(-4 * out[0][2] // 2048) >= tiles
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
