"""First-level rows at the sizes where their building can go wrong: vertex
counts around one sizing tile (256 rows) and one group of tiles (64 tiles),
rows around the eight slots a row is built in, blocks of faces whose vertices
span more than the counting window. Topology is compared exactly with the
oracle; positions within 1e-5 of the bounding-box diagonal (the FP32 bound
every parity test uses)."""
import numpy as np
import pytest

from slak_amd import capi, meshgen as g
from slak_amd.batch import Batch
from slak_amd.mesh import MeshInfo, subdivide_host

pytestmark = pytest.mark.gpu
LAK, SLAK = capi.SLAK_SCHEME_LAK, capi.SLAK_SCHEME_SLAK

SHAPES = {
    "255_vertices": lambda: g.open_grid(14, 16, sigma=1e-3),
    "256_vertices": lambda: g.open_grid(15, 15, sigma=1e-3),
    "257_vertices_valence_256": lambda: g.fan_disk(256),
    "16383_vertices": lambda: g.open_grid(126, 128, sigma=1e-3),
    "16384_vertices": lambda: g.open_grid(127, 127, sigma=1e-3),
    "16385_vertices": lambda: g.open_grid(144, 112, sigma=1e-3),
    "valence_8": lambda: g.uv_sphere(8, 5),
    "valence_9": lambda: g.uv_sphere(9, 5),
    "face_order_8": lambda: g.capped_cylinder(8, 4),
    "face_order_9": lambda: g.capped_cylinder(9, 4),
    "wide_window": lambda: _shuffled(g.torus_mixed(90, 80, 0.3, pentagons=True, seed=3)),
}


def _shuffled(m):
    """The mesh with its vertices renumbered at random (faces far apart in ids)."""
    perm = np.random.default_rng(5).permutation(m.nverts)
    verts = np.empty_like(m.verts)
    verts[perm] = m.verts
    return g.HostMesh(m.type, m.ptr, perm[m.ids].astype(np.int32), m.vals, verts)


def _check(out, ref, diag):
    np.testing.assert_array_equal(out.ids, ref.ids)
    assert np.abs(out.verts.astype(np.float64) - ref.P).max() <= 1e-5 * diag


@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_first_level_rows(oracle, shape, scheme):
    m = SHAPES[shape]()
    out, _ = subdivide_host(m, 1, scheme)
    _check(out, oracle.subdivide(m, 1, scheme=scheme, precision=64), m.bbox_diag())


@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
def test_first_level_rows_in_one_union(oracle, scheme):
    """The same meshes as one batch: mesh bounds inside tiles and groups,
    two replays (the counters start from zero each time)."""
    hosts = [f() for f in SHAPES.values()]
    dev = [MeshInfo.from_host(h) for h in hosts]
    try:
        with Batch(dev, [1] * len(dev), scheme) as b:
            for _ in range(2):
                b.run(use_graph=True)
            for k, h in enumerate(hosts):
                _check(b.result(k).to_host(), oracle.subdivide(h, 1, scheme=scheme, precision=64), h.bbox_diag())
    finally:
        for d in dev:
            d.freeAndReset()
