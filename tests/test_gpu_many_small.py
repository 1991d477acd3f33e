"""Unions in which a block of 256 vertices, faces or corners holds many
meshes, among them meshes without faces, and in which a mesh holds many
blocks: each mesh equals its single-mesh result bit for bit."""
import numpy as np
import pytest

from slak_amd import capi, meshgen as g
from slak_amd.batch import Batch
from slak_amd.mesh import MeshInfo, subdivide_host

pytestmark = pytest.mark.gpu
LAK, SLAK = capi.SLAK_SCHEME_LAK, capi.SLAK_SCHEME_SLAK
NONE = np.zeros(0, np.int32)
KINDS = [g.tetrahedron(), g.cube(), g.torus(5, 4, seed=2), g.open_grid(1, 1, sigma=1e-3), g.open_grid(3, 2, sigma=1e-3),
         g.HostMesh(g.TRI, None, NONE, NONE, np.ones((3, 4), np.float32)), g.torus_mixed(33, 21, 0.3, seed=4)]


@pytest.mark.parametrize("large", [0, 40])
@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
def test_thousands_of_tiny_polygon_meshes(scheme, large):
    """Enough of them that their second level is formed level by level, or,
    beside larger meshes that hold most of the corners, from the input's
    structure; three-level meshes among them."""
    hosts = KINDS[:1] + [g.torus_mixed(40, 30, 0.3, seed=4), g.open_grid(3, 2, sigma=1e-3)]
    kinds = [0] * 3100 + [2] * 50 + [1] * large + [0] * 100
    levels = [2] * (3150 + large) + [3] * 100
    shared = [MeshInfo.from_host(h) for h in hosts]
    try:
        with Batch([shared[k] for k in kinds], levels, scheme) as b:
            for _ in range(2):
                b.run(use_graph=True)
            for i in [0, 1, 77, 3099] + list(range(3100, len(kinds))):
                got, want = b.result(i).to_host(), subdivide_host(hosts[kinds[i]], levels[i], scheme)[0]
                np.testing.assert_array_equal(got.ids, want.ids, err_msg=f"mesh {i}")
                np.testing.assert_array_equal(got.verts.view(np.int32), want.verts.view(np.int32), err_msg=f"mesh {i}")
                if scheme == LAK:
                    np.testing.assert_array_equal(got.ptr, want.ptr, err_msg=f"mesh {i}")
                    np.testing.assert_array_equal(got.vals, want.vals, err_msg=f"mesh {i}")
    finally:
        for d in shared:
            d.freeAndReset()


def draw(name, n):
    if name == "tetrahedra":  # 64 meshes a block of vertices and of faces
        return [0] * n
    rng = np.random.default_rng(7)
    if name == "random":
        return [int(k) for k in rng.integers(0, len(KINDS), n)]
    return [5] * 40 + [6] + [0, 5] * (n // 4) + [5] * 300 + [1] + [5] * 20  # runs of meshes without faces


@pytest.mark.parametrize("levels", [1, 2, 3])
@pytest.mark.parametrize("name", ["tetrahedra", "random", "faceless_runs"])
@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
def test_many_small_meshes(scheme, name, levels):
    kinds = draw(name, 600)
    want = [subdivide_host(h, levels, scheme)[0] for h in KINDS]
    shared = [MeshInfo.from_host(h) for h in KINDS]
    try:
        with Batch([shared[k] for k in kinds], [levels] * len(kinds), scheme) as b:
            b.run(use_graph=True)
            for i, k in enumerate(kinds):
                got = b.result(i).to_host()
                np.testing.assert_array_equal(got.ids, want[k].ids, err_msg=f"mesh {i}")
                np.testing.assert_array_equal(got.verts, want[k].verts, err_msg=f"mesh {i}")
                if scheme == LAK:
                    np.testing.assert_array_equal(got.ptr, want[k].ptr, err_msg=f"mesh {i}")
                    np.testing.assert_array_equal(got.vals, want[k].vals, err_msg=f"mesh {i}")
    finally:
        for d in shared:
            d.freeAndReset()
