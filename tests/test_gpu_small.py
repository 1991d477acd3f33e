"""The first level of a small mesh in one launch against the launches every
other mesh takes (which a mesh of a batch of two takes whatever its size): bit
for bit, at the smallest and largest meshes that are small (1024 vertices and
faces), one vertex or face beyond, rows far longer than their slots, faces
longer than the registers, open and closed meshes, both schemes."""
import numpy as np
import pytest

from slak_amd import capi, meshgen as g
from slak_amd.batch import Batch
from slak_amd.mesh import MeshInfo, subdivide_host

pytestmark = pytest.mark.gpu
LAK, SLAK = capi.SLAK_SCHEME_LAK, capi.SLAK_SCHEME_SLAK

SHAPES = {
    "tetrahedron": g.tetrahedron,
    "cube": g.cube,
    "64_vertices": lambda: g.torus(8, 8, seed=2),
    "65_vertices": lambda: g.torus(13, 5, seed=2),
    "1024_vertices": lambda: g.torus(32, 32, seed=3),
    "1023_vertices": lambda: g.open_grid(30, 32, sigma=1e-3),
    "1025_vertices": lambda: g.open_grid(24, 40, sigma=1e-3),
    "1024_triangles": lambda: g.torus_mixed(32, 16, 1.0, seed=5),
    "1054_triangles": lambda: g.torus_mixed(31, 17, 1.0, seed=5),
    "mixed": lambda: g.torus_mixed(24, 18, 0.3, pentagons=True, seed=4),
    "valence_1000": lambda: g.fan_disk(1000),
    "face_order_300": lambda: g.capped_cylinder(300, 2),
    "polygons": lambda: g.random_poly_torus(13, 11, seed=2),
}


@pytest.mark.parametrize("levels", [1, 3])
@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_small_first_level(shape, scheme, levels):
    m = SHAPES[shape]()
    got, _ = subdivide_host(m, levels, scheme)
    dev = [MeshInfo.from_host(m), MeshInfo.from_host(m)]
    try:
        with Batch(dev, [levels] * 2, scheme) as b:
            b.run()
            want = b.result(1).to_host()
    finally:
        for d in dev:
            d.freeAndReset()
    np.testing.assert_array_equal(got.ids, want.ids)
    np.testing.assert_array_equal(got.verts.view(np.int32), want.verts.view(np.int32))
    if scheme == LAK:
        np.testing.assert_array_equal(got.ptr, want.ptr)
        np.testing.assert_array_equal(got.vals, want.vals)
