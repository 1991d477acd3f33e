"""Levels formed from a polygon mesh two levels back (the output of two
refinements, the positions that deeper meshes go on from) against the
level-by-level chain, bit for bit: triangles to polygons of 300 corners,
valences to 300, open and closed, alone and through the table, both schemes,
and in mixed batches over several replays."""
import numpy as np
import pytest

from slak_amd import capi, meshgen as g
from slak_amd.batch import Batch
from slak_amd.mesh import MeshInfo, subdivide_host

pytestmark = pytest.mark.gpu
LAK, SLAK = capi.SLAK_SCHEME_LAK, capi.SLAK_SCHEME_SLAK

SHAPES = {
    "tetrahedron": g.tetrahedron,
    "tri_9x7": lambda: g.torus_mixed(9, 7, 1.0, seed=5),
    "mixed_40x33": lambda: g.torus_mixed(40, 33, 0.3, pentagons=True, seed=4),
    "polygons": lambda: g.random_poly_torus(13, 11, seed=2),
    "fan_300": lambda: g.fan_disk(300),
    "capped_300": lambda: g.capped_cylinder(300, 2),
    "sphere": lambda: g.uv_sphere(24, 9),
}


def _assert_same(a, b, scheme):
    np.testing.assert_array_equal(a.ids, b.ids)
    np.testing.assert_array_equal(a.verts.view(np.int32), b.verts.view(np.int32))
    if scheme == LAK:
        np.testing.assert_array_equal(a.ptr, b.ptr)
        np.testing.assert_array_equal(a.vals, b.vals)


def _chain(monkeypatch, fn):
    for k in ("SLAK_FUSED_FINAL", "SLAK_FUSED_POS", "SLAK_FINAL_DEEP"):
        monkeypatch.setenv(k, "0")
    out = fn()
    for k in ("SLAK_FUSED_FINAL", "SLAK_FUSED_POS", "SLAK_FINAL_DEEP"):
        monkeypatch.delenv(k)
    return out


@pytest.mark.parametrize("table", ["0", "1"])
@pytest.mark.parametrize("levels", [2, 3, 4])
@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_levels_from_polygons(shape, scheme, levels, table, monkeypatch):
    m = SHAPES[shape]()
    want = _chain(monkeypatch, lambda: subdivide_host(m, levels, scheme)[0])
    monkeypatch.setenv("SLAK_FINAL_TABLE", table)
    _assert_same(subdivide_host(m, levels, scheme)[0], want, scheme)


@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
@pytest.mark.parametrize("deepest", [2, 3, 4, 5])
def test_mixed_batch_from_polygons(scheme, deepest, monkeypatch):
    """Quad, triangle and polygon meshes with depths 1 to deepest (at depth 2
    every mesh ends at the fused level, at 5 one needs the level between),
    three replays; the LAK forms of all depths leave in one launch."""
    hosts = [f() for f in SHAPES.values()] + [g.cube(), g.torus(9, 8, seed=1), g.open_grid(7, 5, sigma=1e-3)]
    levels = [1 + k % deepest for k in range(len(hosts))]
    want = _chain(monkeypatch, lambda: [subdivide_host(h, lv, scheme)[0] for h, lv in zip(hosts, levels)])
    dev = [MeshInfo.from_host(h) for h in hosts]
    try:
        with Batch(dev, levels, scheme) as b:
            for _ in range(3):
                b.run(use_graph=True)
            for k in range(len(hosts)):
                _assert_same(b.result(k).to_host(), want[k], scheme)
    finally:
        for d in dev:
            d.freeAndReset()


@pytest.mark.parametrize("shape", ["closed", "open"])
def test_output_beyond_the_last_level_cache(shape, monkeypatch):
    """More than 224 MiB of positions: k_final's edge points are stored past
    the caches, in whole groups and in the boundary's groups of three."""
    m = g.torus(510, 505, seed=6) if shape == "closed" else g.open_grid(505, 510, sigma=1e-3)
    want = _chain(monkeypatch, lambda: subdivide_host(m, 3, LAK)[0])
    _assert_same(subdivide_host(m, 3, LAK)[0], want, LAK)


@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
def test_two_levels_of_a_mesh_without_faces(scheme):
    """Isolated vertices only: accepted by the level-by-level chain, so not
    handed to the fused level, which has no blocks for it."""
    none = np.zeros(0, np.int32)
    m = g.HostMesh(g.TRI, None, none, none, np.ones((5, 4), np.float32))
    r, _ = subdivide_host(m, 2, scheme)
    assert len(r.verts) == 5 and len(r.ids) == 0
