"""The coarse product c = E^-1 Z^T r of the two-level preconditioner, row for row: one FP64 CG
step moves the iterate by alpha z with z = D^-1 r + Z E^-1 Z^T r, formed here from the oracle's
matrix and the stored E^-1.  Sizes around the points where a row's octets go to one, two or four
waves, a single aggregate, and rows that end inside a group; then a level rebuilt at another
aggregate size against a system that never had another."""
import numpy as np
import pytest
import scipy.sparse as sp

from femocs_amd import fgpu
from femocs_amd import mesh as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu
MARKS = (8, 2, 4, 2)


def _grid(nx, ny, nz):
    """(nx - 1)(ny - 1)(nz - 1) hexes of a jittered box grid, UCD order."""
    X = np.stack(np.meshgrid(*[np.linspace(0.0, n, n) for n in (nx, ny, nz)], indexing="ij"), -1).reshape(-1, 3)
    inner = np.all((X > 0) & (X < [nx, ny, nz]), axis=1)
    X[inner] += np.random.default_rng(3).uniform(-0.2, 0.2, (inner.sum(), 3))
    at = np.arange(nx * ny * nz).reshape(nx, ny, nz)
    lex = np.stack([at[a:nx - 1 + a, b:ny - 1 + b, c:nz - 1 + c].reshape(-1) for c in (0, 1) for b in (0, 1)
                    for a in (0, 1)], 1)
    ucd = np.empty_like(lex)
    ucd[:, M.UCD_TO_LEX] = lex
    return X, ucd.astype(np.int32)


def _system(ctx, X, ucd):
    s = fgpu.System(fgpu.Mesh(ctx, X, ucd, *MARKS))
    s.reset()
    s.add_dirichlet(2, 0.0)
    s.add_neumann(8, None, -1.0)
    s.apply_dirichlet()
    return s


# aggregates: 1, 12 (a row of 16 entries), 512 and 513 (one and two waves), 1024 and 1025 (two and
# four waves, two octets for some lanes of the last)
@pytest.mark.parametrize("shape, agg, nc", [((6, 7, 5), 256, 1), ((14, 15, 14), 256, 12), ((64, 64, 32), 256, 512),
                                            ((64, 64, 33), 256, 528), ((64, 64, 64), 256, 1024),
                                            ((65, 64, 64), 256, 1040), ((64, 64, 33), 512, 264),
                                            ((64, 64, 33), 1024, 132)])
def test_coarse_product_rows(ctx, shape, agg, nc):
    X, ucd = _grid(*shape)
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
    X, ucd = _grid(24, 24, 24)
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
