"""The cut of a mesh's chunks into pieces (charm_mesh_cut, what a context does
with a small mesh): pieces partition the leaves in order within their limits
and their chunk, hold exactly their leaves' faces in (axis, kind) order, every
slot decodes to its leaf's own incidence, and each piece names its chunk's
first leaf."""
import ctypes as C

import numpy as np
import pytest

import charm_3d_amd as CA
import mesh_util as MU


class Pieces(C.Structure):
    _fields_ = [("nch", C.c_int64), ("ncf", C.c_int64)] + \
               [(k, C.POINTER(C.c_int32)) for k in ("eb", "fb", "ref", "cf4")] + [("slots", C.POINTER(C.c_uint16))]


def forest(case):
    if case == "uniform":
        return CA.Forest.uniform(3)
    if case == "adapted":
        return CA.Forest.from_leaves(MU.random_adapted(2, 4, seed=31, frac=0.3))
    return CA.Forest.uniform(1, (True, True, False))


@pytest.mark.parametrize("case", ["uniform", "adapted", "periodic"])
@pytest.mark.parametrize("chunk", [(213, 640), (20, 100)])
@pytest.mark.parametrize("piece", [(8, 48), (48, 192), (1, 6)])
def test_pieces_of_chunks(case, chunk, piece):
    m = forest(case).flatten(*chunk)
    eb0, _, _, sp, _ = m.chunks()
    L, p = CA.lib(), Pieces()
    L.charm_mesh_cut.argtypes = [C.c_void_p, C.c_int, C.c_int, C.POINTER(Pieces)]
    L.charm_pieces_free.argtypes = [C.POINTER(Pieces)]
    CA.check(L.charm_mesh_cut(m.h, *piece, C.byref(p)))
    eb, fb, ref = (np.array(getattr(p, k)[:p.nch + j]) for k, j in (("eb", 1), ("fb", 1), ("ref", 0)))
    cf4, sl = np.array(p.cf4[:4 * p.ncf]).reshape(-1, 4), p.slots[:sp[-1]]
    L.charm_pieces_free(C.byref(p))
    assert eb[0] == 0 and eb[-1] == m.n and (np.diff(eb) > 0).all() and (np.diff(eb) <= piece[0]).all()
    assert fb[0] == 0 and fb[-1] == len(cf4)
    assert ((np.diff(fb) <= piece[1]) | (np.diff(eb) == 1)).all()
    faces = m.faces().tolist()
    rows = {tuple(r): i for i, r in enumerate(faces)}
    inc = [[] for _ in range(m.n)]
    for i, (a, b, _, _) in enumerate(faces):
        inc[a].append((i, 0))
        if b >= 0:
            inc[b].append((i, 1))
    for c in range(len(eb) - 1):
        recs = cf4[fb[c]:fb[c + 1]].tolist()
        ids = [rows[tuple(r)] for r in recs]
        key = [((r[2] & 7) >> 1) * 4 + ((r[2] >> 3) & 3) for r in recs]
        assert len(set(ids)) == len(ids) and key == sorted(key)
        for e in range(eb[c], eb[c + 1]):
            assert sorted((ids[s >> 1], s & 1) for s in sl[sp[e]:sp[e + 1]]) == sorted(inc[e])
        assert set(ids) == {i for e in range(eb[c], eb[c + 1]) for i, _ in inc[e]}
        k = np.searchsorted(eb0, eb[c], side="right") - 1
        assert ref[c] == eb0[k] and eb[c + 1] <= eb0[k + 1]
