"""Batches whose inputs change between runs against their contract (same
topology): the run reports it, and a later run on the restored inputs is as
good as the first."""
import numpy as np
import pytest

from slak_amd import capi, meshgen as g
from slak_amd.batch import Batch
from slak_amd.capi import SlakError
from slak_amd.mesh import MeshInfo

pytestmark = pytest.mark.gpu
LAK, SLAK = capi.SLAK_SCHEME_LAK, capi.SLAK_SCHEME_SLAK


def set_ids(dev, ids):
    ids = np.ascontiguousarray(ids, np.int32)
    capi.check(capi.lib().slak_memcpy_h2d(dev.ids, ids.ctypes.data, ids.nbytes))


def spare_cube():
    """A cube with four unused vertices, and its ids with one face moved to
    them: an open cube and a quad, 16 edges instead of 12."""
    c = g.cube()
    verts = np.concatenate([c.verts, c.verts[:4] + 3.0]).astype(np.float32)
    m = g.HostMesh(g.QUAD, c.ptr, c.ids, c.vals, verts)
    moved = m.ids.copy()
    moved[:4] = [8, 9, 10, 11]
    return m, moved


def assert_same(a, b):
    np.testing.assert_array_equal(a.ids, b.ids)
    np.testing.assert_array_equal(a.verts, b.verts)  # (NaN where NaN: unused vertices)


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
@pytest.mark.parametrize("copies", [1, 3])
@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
def test_an_error_ends_with_its_run(scheme, copies, graph):
    """More edges than planned: that run fails, the next on the original ids
    does not."""
    m, moved = spare_cube()
    dev = [MeshInfo.from_host(m) for _ in range(copies)]
    try:
        with Batch(dev, [1] * copies, scheme) as b:
            b.run(use_graph=graph)
            first = [b.result(k).to_host() for k in range(copies)]
            for _ in range(2):
                set_ids(dev[copies - 1], moved)
                with pytest.raises(SlakError) as ei:
                    b.run(use_graph=graph)
                assert ei.value.code == 5
                set_ids(dev[copies - 1], m.ids)
                b.run(use_graph=graph)
                for k in range(copies):
                    assert_same(b.result(k).to_host(), first[k])
    finally:
        for d in dev:
            d.freeAndReset()
