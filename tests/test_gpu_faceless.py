"""Meshes without faces: vertices alone, which the level chain refines to
themselves. An isolated vertex has valence 0, so its vertex point is 0 / 0 (the
textbook restatement says the same)."""
import numpy as np
import pytest

from slak_amd import capi, meshgen as g
from slak_amd.batch import Batch
from slak_amd.mesh import MeshInfo, subdivide_host

pytestmark = pytest.mark.gpu
LAK, SLAK = capi.SLAK_SCHEME_LAK, capi.SLAK_SCHEME_SLAK


def faceless(kind, nverts=5):
    none = np.zeros(0, np.int32)
    ptr = np.zeros(1, np.int32) if kind == g.POLY else None
    return g.HostMesh(kind, ptr, none, none, np.ones((nverts, 4), np.float32))


def check_faceless(r, nverts):
    assert len(r.ids) == 0 and r.verts.shape == (nverts, 4)
    assert np.isnan(r.verts).all()
    if r.ptr is not None:  # LAK form: no faces, one offset
        np.testing.assert_array_equal(r.ptr, [0])


@pytest.mark.parametrize("kind", [g.TRI, g.POLY], ids=["tri", "poly"])
@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
@pytest.mark.parametrize("nverts", [1, 5, 256, 1500])
def test_two_levels_without_corner_items(scheme, kind, nverts):
    """The second level's row offsets end with the last vertex item: no corner
    item runs in a union without faces."""
    m = faceless(kind, nverts)
    for _ in range(3):  # on recycled memory too
        subdivide_host(g.torus(9, 7), 3, scheme)
        check_faceless(subdivide_host(m, 2, scheme)[0], nverts)


@pytest.mark.parametrize("table", ["0", "1"])
@pytest.mark.parametrize("levels", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("kind", [g.TRI, g.POLY, g.QUAD], ids=["tri", "poly", "quad"])
@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
def test_alone_at_every_depth(scheme, kind, levels, table, monkeypatch):
    """Accepted at one level, so at every level: the last level's launch has
    vertex blocks alone."""
    monkeypatch.setenv("SLAK_FINAL_TABLE", table)
    check_faceless(subdivide_host(faceless(kind), levels, scheme)[0], 5)


@pytest.mark.parametrize("levels", [2, 3, 4, 5])
@pytest.mark.parametrize("others", ["open", "closed", "none"])
@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
def test_in_a_batch(scheme, others, levels):
    """Beside open meshes alone (no mesh of the batch then comes from three
    levels back), beside closed ones, and beside other meshes without faces."""
    rest = {"open": [g.open_grid(5, 4, sigma=1e-3)], "closed": [g.cube(), g.torus_mixed(8, 6, 0.3, seed=2)],
            "none": [faceless(g.QUAD, 300)]}[others]
    hosts = [faceless(g.TRI), *rest, faceless(g.POLY, 9)]
    dev = [MeshInfo.from_host(h) for h in hosts]
    try:
        with Batch(dev, [levels] * len(hosts), scheme) as b:
            for graph in (False, True):
                b.run(use_graph=graph)
                check_faceless(b.result(0).to_host(), 5)
                check_faceless(b.result(len(hosts) - 1).to_host(), 9)
                for k, h in enumerate(rest):
                    got, want = b.result(1 + k).to_host(), subdivide_host(h, levels, scheme)[0]
                    np.testing.assert_array_equal(got.ids, want.ids)
                    np.testing.assert_array_equal(got.verts, want.verts)
    finally:
        for d in dev:
            d.freeAndReset()
