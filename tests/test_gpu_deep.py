"""The output level formed from three levels back (closed LAK meshes of four
levels or more) against the output level from two levels back, which the other
tests compare with the level-by-level chain and the oracle: bit for bit, alone
and in mixed batches, at work-unit edges (a few faces, valences from 3 to 24,
polygons) and through both descriptor paths."""
import numpy as np
import pytest

from slak_amd import capi, meshgen as g
from slak_amd.batch import Batch
from slak_amd.mesh import MeshInfo, subdivide_host

pytestmark = pytest.mark.gpu
LAK = capi.SLAK_SCHEME_LAK

CLOSED = {
    "cube": g.cube,
    "tetrahedron": g.tetrahedron,
    "torus_5x4": lambda: g.torus(5, 4, seed=2),
    "torus_17x13": lambda: g.torus(17, 13, seed=3),
    "mixed_24x18": lambda: g.torus_mixed(24, 18, 0.3, pentagons=True, seed=4),
    "tri_9x7": lambda: g.torus_mixed(9, 7, 1.0, seed=5),
    "sphere_24x4": lambda: g.uv_sphere(24, 4),
    "capped_9x3": lambda: g.capped_cylinder(9, 3),
}


def _assert_same(a, b):
    np.testing.assert_array_equal(a.ids, b.ids)
    np.testing.assert_array_equal(a.verts.view(np.int32), b.verts.view(np.int32))
    np.testing.assert_array_equal(a.ptr, b.ptr)
    np.testing.assert_array_equal(a.vals, b.vals)


@pytest.mark.parametrize("table", ["0", "1"])
@pytest.mark.parametrize("levels", [4, 5])
@pytest.mark.parametrize("shape", list(CLOSED))
def test_output_level_from_three_levels_back(shape, levels, table, monkeypatch):
    m = CLOSED[shape]()
    monkeypatch.setenv("SLAK_FINAL_DEEP", "0")
    want, _ = subdivide_host(m, levels, LAK)
    monkeypatch.delenv("SLAK_FINAL_DEEP")
    monkeypatch.setenv("SLAK_FINAL_TABLE", table)
    got, _ = subdivide_host(m, levels, LAK)
    _assert_same(got, want)


def test_mixed_batch_with_deep_meshes(monkeypatch):
    """Depths 1 to 5, open meshes among the closed ones (the boundary variants
    of the other kernels then run on the same levels), three replays."""
    hosts = [f() for f in CLOSED.values()] + [g.open_grid(7, 5, sigma=1e-3), g.fan_disk(11), g.torus(6, 6, seed=9),
                                              g.torus_mixed(12, 9, 0.2, seed=8), g.random_poly_torus(13, 11, seed=2)]
    levels = [4, 5, 4, 4, 4, 5, 4, 4, 4, 5, 1, 2, 3]
    monkeypatch.setenv("SLAK_FINAL_DEEP", "0")
    want = [subdivide_host(h, lv, LAK)[0] for h, lv in zip(hosts, levels)]
    monkeypatch.delenv("SLAK_FINAL_DEEP")
    dev = [MeshInfo.from_host(h) for h in hosts]
    try:
        with Batch(dev, levels, LAK) as b:
            for _ in range(3):
                b.run(use_graph=True)
            for k in range(len(hosts)):
                _assert_same(b.result(k).to_host(), want[k])
    finally:
        for d in dev:
            d.freeAndReset()


def test_output_beyond_the_last_level_cache(monkeypatch):
    """276 MB of positions: the edge points are stored past the caches."""
    m = g.torus(270, 250, seed=6)
    monkeypatch.setenv("SLAK_FINAL_DEEP", "0")
    want, _ = subdivide_host(m, 4, LAK)
    monkeypatch.delenv("SLAK_FINAL_DEEP")
    got, _ = subdivide_host(m, 4, LAK)
    _assert_same(got, want)
