"""Per-dof kernels with one dof per thread (small systems) and four: solves on both sides of the
limit and around whole workgroups agree with the oracle, alone and in one batch bit for bit, and a
level of larger aggregates takes a small system back to four."""
import numpy as np
import pytest

from box_grid import box_grid
from femocs_amd import fgpu
from oracle import oracle as O

pytestmark = pytest.mark.gpu
MARKS = (8, 2, 4, 2)


def _system(ctx, X, ucd, agg):
    s = fgpu.System(fgpu.Mesh(ctx, X, ucd, *MARKS))
    s.reset()
    s.add_dirichlet(2, 0.0)
    s.add_neumann(8, None, -1.0)
    s.apply_dirichlet()
    if agg:
        s.set_coarse(agg)
    return s


@pytest.mark.parametrize("precision, agg", [(fgpu.FGPU_FP64, 0), (fgpu.FGPU_MIXED, 0), (fgpu.FGPU_FP64, 256),
                                            (fgpu.FGPU_MIXED, 256), (fgpu.FGPU_MIXED, 512), (fgpu.FGPU_MIXED, 1024)])
def test_solves_around_the_limits(ctx, precision, agg):
    # 256 dofs (one workgroup), 258, 1028 (four workgroups and 4 dofs); 49152 (the last small size)
    # and 49248
    shapes = [(8, 8, 4), (2, 3, 43), (257, 2, 2), (48, 32, 32), (48, 27, 38)]
    o = fgpu.opts(tol=1e-12, precision=precision, inner_tol=0.01)
    systems, alone = [], []
    for shape in shapes:
        X, ucd = box_grid(*shape)
        s = _system(ctx, X, ucd, agg)
        s.fill_solution(0.0)
        st = s.solve(o)
        _, ref, it, _, _ = O.poisson_laplace(X, ucd, -1.0, tol=1e-13, relative=True)
        assert st.iterations > 0 and it > 0
        x = s.solution()
        assert np.linalg.norm(x - ref) <= 1e-10 * np.linalg.norm(ref)
        systems.append(s)
        alone.append((st.iterations, x))
    for s in systems:
        s.fill_solution(0.0)
    stats = ctx.solve_batch(systems, o)
    for s, st, (it, x) in zip(systems, stats, alone):
        assert st.iterations == it and np.array_equal(s.solution(), x)


@pytest.mark.parametrize("precision", [fgpu.FGPU_FP64, fgpu.FGPU_MIXED])
@pytest.mark.parametrize("drop", ["off", "refused"])
def test_dropped_level_leaves_no_trace(ctx, precision, drop):
    """A small system whose level of larger aggregates was dropped gives the bits of one that
    never had a level."""
    X, ucd = box_grid(24, 24, 24)
    o = fgpu.opts(tol=1e-10, precision=precision, inner_tol=0.01)
    out = []
    for before in (False, True):
        s = _system(ctx, X, ucd, 1024 if before else 0)
        if before and drop == "off":
            s.set_coarse(False)
        elif before:
            with pytest.raises(fgpu.FgpuError):
                s.set_coarse(77)
        s.fill_solution(0.0)
        out.append((s.solve(o).iterations, s.solution()))
    assert out[0][0] > 0 and out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
