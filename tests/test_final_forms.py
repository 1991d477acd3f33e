"""The closed forms of the last levels' kernels (slak_amd/csrc/slak_kernels.hip)
against brute force on the refined meshes: the output level from a polygon mesh
two levels back (final_corner, final_face), and from a closed quad mesh three
levels back (deep_corner, deep_edges)."""
import numpy as np
import pytest

from slak_amd import meshgen as g
from tests import structure_model as M

POLYGONS = [
    ("tetrahedron", lambda: g.tetrahedron()),
    ("cube", lambda: g.cube()),
    ("open_grid", lambda: g.open_grid(5, 3, sigma=0.01)),
    ("fan", lambda: g.fan_disk(7)),
    ("capped", lambda: g.capped_cylinder(9, 2)),
    ("mixed_pent", lambda: g.torus_mixed(12, 8, 0.3, pentagons=True, seed=7)),
    ("mixed_tri", lambda: g.torus_mixed(9, 7, 0.5, seed=3)),
    ("random", lambda: g.random_poly_torus(7, 6, seed=2)),
]




@pytest.mark.parametrize("name,make", POLYGONS, ids=[m[0] for m in POLYGONS])
@pytest.mark.parametrize("scheme", [M.LAK, M.SLAK], ids=["LAK", "SLAK"])
def test_output_level_from_polygons(name, make, scheme):
    mesh = make()
    S = M.structure_of(mesh.face_ptr(), mesh.ids, mesh.nverts, scheme)
    S1 = M.refine_structure(S, scheme)
    brute = M.structure_of(np.arange(len(S1.ids) // 4 + 1) * 4, S1.ids, S1.nv, scheme)
    cface, nextc, prevc = M._corner_tables(S.ptr)
    nv, nf, nnz, ne = S.nv, len(S.ptr) - 1, len(S.ids), len(S.bnd)
    ep0, nv1 = nv + nf, nv + nf + ne
    blk = np.concatenate([[0], np.cumsum(S.bnd)]).astype(np.int64)
    rows = lambda v: brute.rows[int(brute.tptr[v]):int(brute.tptr[v + 1])]
    written = {}
    for t in range(nnz):
        F, tn, tp = int(cface[t]), int(nextc[t]), int(prevc[t])
        v, w, u = int(S.ids[t]), int(S.ids[tn]), int(S.ids[tp])
        e1, e0, s1, s0 = int(S.eout[t]), int(S.eout[tp]), int(S.twin[t]), int(S.twin[tp])
        g1, n1, p1 = (int(cface[s1]), int(nextc[s1]), int(prevc[s1])) if s1 >= 0 else (F, 0, 0)
        g0 = int(cface[s0]) if s0 >= 0 else F
        if scheme == M.LAK:
            b1, b0 = 4 * e1 - int(blk[e1]), 4 * e0 - int(blk[e0])
            E1 = [b1 + (v > w), b1 + 2 + (s1 >= 0 and F > g1), b0 + 2 + (s0 >= 0 and F > g0), b0 + (v > u)]
        else:
            E1 = [int(S.mpos[t]), nnz + tn, nnz + t, 2 * nnz + int(blk[e0]) if s0 < 0 else int(S.mpos[s0])]
        # M1 face t and the ids of its edges
        assert list(S1.ids[4 * t: 4 * t + 4]) == [v, ep0 + e1, nv + F, ep0 + e0]
        assert [int(x) for x in brute.eout[4 * t: 4 * t + 4]] == [int(x) for x in E1]
        if not (s1 < 0 or t < s1):
            continue
        # the owner of e1: its M1 edges, once each, and the row of ep(e1)
        if scheme == M.LAK:
            out = {4 * t: b1 + (v > w), 4 * tn + 3: b1 + (w > v), 4 * t + 1: b1 + 2 + (s1 >= 0 and F > g1)}
            if s1 >= 0:
                out[4 * s1 + 1] = b1 + 2 + (g1 > F)
        else:
            out = {4 * t: int(S.mpos[t]), 4 * tn + 3: int(S.mpos[s1]) if s1 >= 0 else 2 * nnz + int(blk[e1]),
                   4 * t + 1: nnz + tn}
            if s1 >= 0:
                out[4 * s1 + 1] = nnz + n1
        for c, e in out.items():
            assert int(brute.eout[c]) == e and e not in written
            written[e] = c
        ent = [(4 * t + 1, v), (4 * tn + 3, nv + F)]
        if s1 >= 0:
            ent += [(4 * s1 + 1, w), (4 * n1 + 3, nv + g1)]
            # the M1 faces of the twin and of the corner after it
            assert list(S1.ids[4 * s1: 4 * s1 + 4]) == [w, ep0 + e1, nv + g1, ep0 + int(S.eout[p1])]
            assert list(S1.ids[4 * n1: 4 * n1 + 4]) == [v, ep0 + int(S.eout[n1]), nv + g1, ep0 + e1]
        assert rows(ep0 + e1) == sorted(ent)
    assert sorted(written) == list(range(len(S1.bnd)))
    for F in range(nf):
        corners = range(int(S.ptr[F]), int(S.ptr[F + 1]))
        assert rows(nv + F) == [(4 * t + 2, ep0 + int(S.eout[t])) for t in corners]


CLOSED = [
    ("cube", lambda: g.cube()),
    ("torus_5x4", lambda: g.torus(5, 4, seed=2)),
    ("tetrahedron_l1", lambda: g.tetrahedron()),
    ("mixed_l1", lambda: g.torus_mixed(6, 5, 0.3, pentagons=True, seed=7)),
    ("capped_l1", lambda: g.capped_cylinder(5, 2)),
]


@pytest.mark.parametrize("name,make", CLOSED, ids=[m[0] for m in CLOSED])
def test_output_level_from_three_levels_back(name, make):
    mesh = make()
    N = M.structure_of(mesh.face_ptr(), mesh.ids, mesh.nverts, M.LAK)
    if mesh.type != g.QUAD:
        N = M.refine_structure(N, M.LAK)
    Ms = M.refine_structure(N, M.LAK)
    M1 = M.structure_of(np.arange(len(Ms.ids) + 1) * 4, M.refine_structure(Ms, M.LAK).ids,
                        M.refine_structure(Ms, M.LAK).nv, M.LAK)
    nv, nf, nnz, ne = N.nv, len(N.ids) // 4, len(N.ids), len(N.bnd)
    assert 2 * ne == nnz
    epN = nv + nf
    fM = epN + ne
    eM = fM + nnz
    # M's corners from N's
    for t in range(nnz):
        f, q0 = t >> 2, t & ~3
        tn, tp = q0 | ((t + 1) & 3), q0 | ((t + 3) & 3)
        v, w, u = int(N.ids[t]), int(N.ids[tn]), int(N.ids[tp])
        e1, e0, s1, s0 = int(N.eout[t]), int(N.eout[tp]), int(N.twin[t]), int(N.twin[tp])
        n1 = (s1 & ~3) | ((s1 + 1) & 3)
        assert list(Ms.ids[4 * t: 4 * t + 4]) == [v, epN + e1, nv + f, epN + e0]
        assert [int(x) for x in Ms.eout[4 * t: 4 * t + 4]] == [
            4 * e1 + (v > w), 4 * e1 + 2 + (f > s1 >> 2), 4 * e0 + 2 + (f > s0 >> 2), 4 * e0 + (v > u)]
        assert [int(x) >> 2 for x in Ms.twin[4 * t: 4 * t + 4]] == [n1, tn, tp, s0]
    # the rows of 16 lanes around every N edge
    face_of = {frozenset(int(x) for x in M1.ids[4 * i: 4 * i + 4]): i for i in range(len(M1.ids) // 4)}
    edge_id = {}
    for c in range(len(M1.ids)):
        edge_id[frozenset((int(M1.ids[c]), int(M1.ids[(c & ~3) | ((c + 1) & 3)])))] = int(M1.eout[c])
    row = lambda x: M1.rows[int(M1.tptr[x]):int(M1.tptr[x + 1])]
    for t in range(nnz):
        s = int(N.twin[t])
        if t > s:
            continue
        e = int(N.eout[t])
        v, w, f, h = int(N.ids[t]), int(N.ids[s]), t >> 2, s >> 2
        nxt = lambda c: (c & ~3) | ((c + 1) & 3)
        A = [v, nv + f, w, nv + h]
        Z = [fM + t, fM + nxt(t), fM + s, fM + nxt(s)]
        Y = [4 * e + (v > w), 4 * e + 2, 4 * e + (w > v), 4 * e + 3]
        X = epN + e
        tt, ss = (t & 3) != 3, (s & 3) != 3
        psi = {}
        for j in range(4):
            jp, jn = (j + 3) & 3, (j + 1) & 3
            y = eM + Y[j]
            zfirst = j == 0 or (j == 1 and not tt) or (j == 3 and not ss)
            nbr = [A[j], Z[j], X, Z[jp]]
            slot = [0, 2 if zfirst else 3, 1, 3 if zfirst else 2]
            for m in range(4):
                assert edge_id[frozenset((nbr[m], y))] == 4 * Y[j] + slot[m], (j, m)
            # faces after each neighbour; the ones at A_j hold another M edge of A_j
            around = [r[0] >> 2 for r in row(y)]
            assert len(around) == 4
            psi[j, 1] = face_of[frozenset((X, eM + Y[jn], Z[j], y))]
            psi[j, 2] = face_of[frozenset((X, y, Z[jp], eM + Y[jp]))]
            at_a = [x for x in around if A[j] in M1.ids[4 * x: 4 * x + 4]]
            psi[j, 0] = next(x for x in at_a if Z[j] in M1.ids[4 * x: 4 * x + 4])
            psi[j, 3] = next(x for x in at_a if Z[jp] in M1.ids[4 * x: 4 * x + 4])
            odd = j & 1
            first = [psi[j, 0], psi[j, 1]]          # corners in Z_j: A_j's first
            second = [psi[j, 2], psi[j, 3]] if odd else [psi[j, 3], psi[j, 2]]
            assert around == (first + second if zfirst else second + first)
            n0, n1 = (X, Z[jp]) if odd else (Z[jp], X)
            assert [r[1] for r in row(y)] == ([A[j], Z[j], n0, n1] if zfirst else [n0, n1, A[j], Z[j]])
        a, b = (0, 1) if tt else (1, 0)
        c, d = (2, 3) if ss else (3, 2)
        assert [r[0] >> 2 for r in row(X)] == [psi[j, 1] for j in (a, b, c, d)]
        assert [r[1] for r in row(X)] == [eM + Y[j] for j in (a, b, c, d)]


@pytest.mark.parametrize("name,make", POLYGONS + CLOSED[:1], ids=[m[0] for m in POLYGONS + CLOSED[:1]])
def test_boundary_ranks_of_the_refined_mesh(name, make):
    """The boundary edges before each refined edge, as the owners of the edges
    hand them on (LAK), over two refinements."""
    mesh = make()
    S = M.structure_of(mesh.face_ptr(), mesh.ids, mesh.nverts, M.LAK)
    for _ in range(2):
        S1 = M.refine_structure(S, M.LAK)
        blk = np.concatenate([[0], np.cumsum(S.bnd)]).astype(np.int64)
        got = np.full(len(S1.bnd), -1, dtype=np.int64)
        for e in range(len(S.bnd)):
            b, bl = int(S.bnd[e] != 0), int(blk[e])
            ranks = [2 * bl, 2 * bl + b, 2 * bl + 2 * b] + ([] if b else [2 * bl])
            got[4 * e - bl: 4 * e - bl + len(ranks)] = ranks
        np.testing.assert_array_equal(got, np.concatenate([[0], np.cumsum(S1.bnd)])[:-1])
        S = S1
