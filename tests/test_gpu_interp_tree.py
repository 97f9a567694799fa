"""Point search on trees of every small size (one leaf, two, ...) and across the sizes of a call
(16 lanes share a point up to 32768 points, 8 above, one above 131072): located cells equal the
oracle's scan, on either build of the tables, and the same points in one call of each kind give
the same cells."""
from types import SimpleNamespace

import numpy as np
import pytest

from femocs_amd import interp
from femocs_amd import mesh as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _part(small_mesh, k):
    """The first k tets of the mesh around its middle, as a mesh of their own, split into hexes."""
    c = small_mesh.nodes[small_mesh.tets].mean(1)
    pick = np.argsort(np.linalg.norm(c - c.mean(0), axis=1), kind="stable")[:k]
    used, tets = np.unique(small_mesh.tets[pick], return_inverse=True)
    tets = tets.reshape(-1, 4)
    nodes, kind, hexes = M.tet_to_hex(small_mesh.nodes[used], tets)
    marker = np.where(np.arange(k) % 4 == 3, M.TYPES_BULK, M.TYPES_VACUUM).astype(np.int32)
    hm = np.where(np.repeat(marker, 4) == M.TYPES_VACUUM, 1, -1).astype(np.int32)
    return SimpleNamespace(nodes=nodes, node_kind=kind, tets=tets.astype(np.int32), tet_marker=marker,
                           tet_nbr=M._face_neighbours(tets), hexes=hexes, hex_marker=hm)


@pytest.mark.parametrize("host_build", [False, True])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 7, 64, 65, 300])
@pytest.mark.parametrize("n", [1, 65, 2500, 32769])
def test_located_cells(ctx, small_mesh, host_build, k, n):
    part = _part(small_mesh, k)
    ip = interp.Interpolator(ctx, part, interp.TYPES_VACUUM, host_build=host_build)
    L = O.LinTet(part.nodes, part.tets, part.tet_nbr, part.tet_marker, 3)
    rng = np.random.default_rng(100 * k + n)
    P = part.nodes[part.tets]
    t = rng.integers(0, k, n)
    inside = (P[t] * rng.dirichlet(np.ones(4), n)[:, :, None]).sum(1)
    lo, hi = part.nodes.min(0), part.nodes.max(0)
    anywhere = rng.uniform(lo - 0.3 * (hi - lo), hi + 0.3 * (hi - lo), (n, 3))
    pts = np.where(rng.random(n)[:, None] < 0.5, inside, anywhere)
    pts[:: 7] = P[t[::7], 0]                       # on vertices: several cells hold the point
    ip.set_nodal(rng.standard_normal((len(part.nodes), 5)))
    cells, _ = ip.points(pts, 1)
    ref, _ = O.interp_points(L, part.nodes, part.tets, O.quadtet_cells(part.tets, part.hexes, part.node_kind),
                             part.hexes, ip.nodal(), pts, 1)
    assert np.array_equal(cells, ref)


def test_lanes_per_point_find_the_same_cells(ctx, small_mesh):
    ip = interp.Interpolator(ctx, small_mesh, interp.TYPES_VACUUM)
    rng = np.random.default_rng(8)
    lo, hi = small_mesh.nodes.min(0), small_mesh.nodes.max(0)
    pts = rng.uniform(lo - 0.05 * (hi - lo), hi + 0.05 * (hi - lo), (131073, 3))
    pts[::5] = small_mesh.nodes[rng.integers(0, len(small_mesh.nodes), len(pts[::5]))]
    ip.set_nodal(np.zeros((len(small_mesh.nodes), 5)))
    one = ip.points(pts, 1)[0]
    for n in (131072, 32768, 777):
        assert np.array_equal(ip.points(pts[:n], 1)[0], one[:n])


@pytest.mark.parametrize("rank", [1, 3])
def test_lanes_per_point_find_the_same_faces(ctx, small_mesh, rank):
    """The surface search (faces and the tets behind them) at one, 8 and 16 lanes a point: the chain
    of a call's first points is that of a shorter call, also with atoms on face vertices and edges,
    which lie in several faces."""
    tip = small_mesh
    tris, t2t = tip.surface_triangles()
    ip = interp.Interpolator(ctx, tip, interp.TYPES_VACUUM)
    ip.set_triangles(tris, t2t, tip.surface_quads(tris))
    rng = np.random.default_rng(21)
    ip.set_nodal(rng.standard_normal((len(tip.nodes), 5)))
    n = 131073
    w = rng.dirichlet(np.ones(3), n)
    w[::5] = np.eye(3)[rng.integers(0, 3, len(w[::5]))]              # vertices
    w[1::5, 0], w[1::5, 1], w[1::5, 2] = 0.5, 0.5, 0.0               # edge centres
    pts = np.einsum("nk,nkd->nd", w, tip.nodes[tris[rng.integers(0, len(tris), n)]])
    pts[2::5] += rng.normal(0.0, 0.3, pts[2::5].shape)               # off the surface
    one, val = ip.surface_points(pts, rank)
    assert (one < 0).any() and (one > 0).any()
    for m in (131072, 32769, 32768, 777):
        cells, out = ip.surface_points(pts[:m], rank)
        assert np.array_equal(cells, one[:m]) and np.array_equal(out, val[:m])
