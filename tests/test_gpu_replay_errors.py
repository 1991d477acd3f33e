"""Errors of the first level's analysis: what a call on an invalid mesh reports,
and batches whose inputs change between runs against their contract (same
topology): the run reports it, and a later run on the restored inputs is as
good as the first."""
import ctypes

import numpy as np
import pytest

from slak_amd import capi, meshgen as g
from slak_amd.batch import Batch
from slak_amd.capi import SlakError
from slak_amd.mesh import LAKCatmullClark, MeshInfo, subdivide_host

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


def changed(kind):
    """A mesh and ids that break the contract: (mesh, other ids, flag text)."""
    if kind == "more_edges":
        m, ids = spare_cube()
        return m, ids, "number of edges"
    if kind == "fewer_edges":  # the open cube and the quad become the cube
        m, ids = spare_cube()
        return g.HostMesh(m.type, m.ptr, ids, m.vals, m.verts), m.ids, "number of edges"
    m = g.uv_sphere(12, 5)  # rows beyond their eight slots
    ids = m.ids.copy()
    if kind == "bad_id":
        ids[5] = m.nverts
        return m, ids, "vertex id out of range"
    assert kind == "turned_face"
    ids[:3] = ids[:3][::-1]
    return m, ids, "non-manifold"


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
@pytest.mark.parametrize("levels", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("kind", ["more_edges", "fewer_edges", "bad_id", "turned_face"])
@pytest.mark.parametrize("scheme", [LAK, SLAK], ids=["LAK", "SLAK"])
def test_nothing_is_refined_from_a_failed_analysis(scheme, kind, levels, graph):
    """Changed before the first run (nothing a level reads has been written
    then) and after a good one: the run reports the flag, the kernels after the
    analysis write nothing, and the original ids give the same result again.
    Alone and between other meshes."""
    m, ids, text = changed(kind)
    want = subdivide_host(m, levels, scheme)[0]
    for hosts in ([m], [g.torus(6, 5, seed=2), m, g.open_grid(4, 3, sigma=1e-3)]):
        at = len(hosts) // 2
        dev = [MeshInfo.from_host(h) for h in hosts]
        try:
            with Batch(dev, [levels] * len(hosts), scheme) as b:
                for again in range(2):
                    set_ids(dev[at], ids)
                    before = [b.result(k).to_host() for k in range(len(hosts))]
                    with pytest.raises(SlakError) as ei:
                        b.run(use_graph=graph)
                    assert ei.value.code == 5 and text in str(ei.value)
                    if again and levels > 1:
                        for k in range(len(hosts)):
                            assert_same(b.result(k).to_host(), before[k])
                    set_ids(dev[at], m.ids)
                    b.run(use_graph=graph)
                    assert_same(b.result(at).to_host(), want)
        finally:
            for d in dev:
                d.freeAndReset()


@pytest.mark.parametrize("shape", ["small", "launches"])
@pytest.mark.parametrize("kind", ["bad_id", "turned_face"])
def test_an_error_names_its_mesh_on_any_stream(kind, shape):
    """The flags of each mesh are read after the kernel that writes them, also
    on a stream that copies do not wait for."""
    m = g.uv_sphere(12, 5) if shape == "small" else g.uv_sphere(12, 200)
    ids = m.ids.copy()
    ids[:3] = (m.nverts, ids[1], ids[2]) if kind == "bad_id" else ids[:3][::-1]
    text = "vertex id out of range" if kind == "bad_id" else "non-manifold"
    bad = MeshInfo.from_host(g.HostMesh(m.type, m.ptr, ids, m.vals, m.verts))
    st = ctypes.c_void_p()
    assert capi.lib().hipStreamCreateWithFlags(ctypes.byref(st), ctypes.c_uint(1)) == 0  # non-blocking
    try:
        for _ in range(20):
            with pytest.raises(SlakError) as ei:
                LAKCatmullClark.subdivideIteratively(bad, MeshInfo(), 2, st.value)
            assert ei.value.code == 2 and "mesh 0:" in str(ei.value) and text in str(ei.value)
    finally:
        capi.lib().hipStreamDestroy(st)
        bad.freeAndReset()
