"""Meshes without faces: vertices alone, which the level chain refines to
themselves. An isolated vertex has valence 0, so its vertex point is 0 / 0 (the
textbook restatement says the same)."""
import numpy as np
import pytest

from slak_amd import capi, meshgen as g
from slak_amd.mesh import subdivide_host

pytestmark = pytest.mark.gpu
LAK, SLAK = capi.SLAK_SCHEME_LAK, capi.SLAK_SCHEME_SLAK


def faceless(kind, nverts=5):
    none = np.zeros(0, np.int32)
    ptr = np.zeros(1, np.int32) if kind == g.POLY else None
    return g.HostMesh(kind, ptr, none, none, np.ones((nverts, 4), np.float32))


def check_faceless(r, nverts):
    assert len(r.ids) == 0 and r.verts.shape == (nverts, 4)
    assert np.isnan(r.verts).all()


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
