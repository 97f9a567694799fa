"""The coarse product c = E^-1 Z^T r of the two-level preconditioner, row for row: one FP64 CG
step moves the iterate by alpha z with z = D^-1 r + Z E^-1 Z^T r, formed here from the oracle's
matrix and the stored E^-1.  Sizes around the points where a row's octets go to one, two or four
waves, a single aggregate, and rows that end inside a group; then a level rebuilt at another
aggregate size against a system that never had another."""
import numpy as np
import pytest
import scipy.sparse as sp

from box_grid import box_grid
from femocs_amd import fgpu
from oracle import oracle as O

pytestmark = pytest.mark.gpu
MARKS = (8, 2, 4, 2)


def _system(ctx, X, ucd):
    s = fgpu.System(fgpu.Mesh(ctx, X, ucd, *MARKS))
    s.reset()
    s.add_dirichlet(2, 0.0)
    s.add_neumann(8, None, -1.0)
    s.apply_dirichlet()
    return s


# aggregates: 1; 5, 6 and 7 (the last group of four rows holds 1, 2 and 3); 12 (a row of 16 entries);
# 512 and 513 (one and two waves a group, 513 ends in a group of one row), 528; 1024 and 1025 (two and
# four waves, two octets for some lanes of the last), 1040; larger aggregates, 257 of 512 dofs and 129
# of 1024 in a cut group
@pytest.mark.parametrize("shape, agg, nc", [((6, 7, 5), 256, 1), ((14, 15, 14), 256, 12), ((64, 64, 32), 256, 512),
                                            ((9, 10, 12), 256, 5), ((9, 11, 13), 256, 6), ((10, 12, 13), 256, 7),
                                            ((41, 50, 64), 256, 513), ((41, 79, 81), 256, 1025),
                                            ((41, 50, 64), 512, 257), ((41, 50, 64), 1024, 129),
                                            ((64, 64, 33), 256, 528), ((64, 64, 64), 256, 1024),
                                            ((65, 64, 64), 256, 1040), ((64, 64, 33), 512, 264),
                                            ((64, 64, 33), 1024, 132)])
def test_coarse_product_rows(ctx, shape, agg, nc):
    X, ucd = box_grid(*shape, jitter=0.2)
    s = _system(ctx, X, ucd)
    s.set_coarse(agg)
    block, einv = s.coarse()
    assert len(einv) == nc
    om = O.Mesh(X, ucd, *MARKS)
    om.assemble()
    b = om.face_rhs(8, constant=-1.0)
    mask = om.dirichlet_mask(2)
    om.apply_dirichlet(b, np.zeros(om.n_dofs), mask, None)
    rp, ci, va = om.csr()
    A = sp.csr_matrix((va, ci, rp), shape=(om.n_dofs, om.n_dofs))
    free = mask == 0
    x0 = np.random.default_rng(nc).standard_normal(om.n_dofs) * free
    r = (b - A @ x0) * free
    Z = sp.csr_matrix((free.astype(float), (np.arange(om.n_dofs), block)), shape=(om.n_dofs, nc))
    z = free * (r / A.diagonal()) + Z @ (einv.astype(np.float64) @ (Z.T @ r))
    step = (r @ z) / (z @ (A @ z)) * z
    s.set_solution(x0)
    s.solve(fgpu.opts(tol=1e-14, max_it=1, use_graph=False))
    # sums of up to nc products in another order: rounding of about sqrt(nc) eps, cancellation in r
    assert np.linalg.norm(s.solution() - x0 - step) <= 1e-12 * np.linalg.norm(step)


@pytest.mark.parametrize("precision", [fgpu.FGPU_FP64, fgpu.FGPU_MIXED])
def test_coarse_level_rebuilt_at_another_size(ctx, precision):
    """The partial sums of the smaller aggregates must not stay in the larger ones' r.z."""
    X, ucd = box_grid(24, 24, 24, jitter=0.2)
    o = fgpu.opts(tol=1e-10, precision=precision, inner_tol=0.01)
    out = []
    for sizes in ((1024,), (256, 1024)):
        s = _system(ctx, X, ucd)
        for agg in sizes:
            s.set_coarse(agg)
            s.fill_solution(0.0)
            st = s.solve(o)
        out.append((st.iterations, s.solution()))
    assert out[0][0] > 0 and out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
