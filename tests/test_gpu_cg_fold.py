"""Folded CG iterations (the element apply and the vector kernel sum the partials themselves)
against iterations with scalar kernels: a system gives the same bits and iteration counts either
way.  A solve alone folds; in a batch with a tip above the patch limit the same system does not."""
import numpy as np
import pytest

from femocs_amd import fgpu, serving
from femocs_amd import mesh as M

pytestmark = pytest.mark.gpu
MARKS = (8, 2, 4, 2)


def _system(ctx, tip, cells, coarse):
    gm = fgpu.Mesh(ctx, tip.nodes, tip.vacuum_cells(), *MARKS)
    if cells:
        gm.set_patch_cells(cells)
    s = fgpu.System(gm)
    s.reset()
    s.add_dirichlet(2, 0.0)
    s.add_neumann(8, None, -1.0)
    s.apply_dirichlet()
    if coarse:
        s.set_coarse(True)
    return s


@pytest.mark.parametrize("precision, coarse, precond", [
    (fgpu.FGPU_FP64, False, fgpu.FGPU_PC_JACOBI), (fgpu.FGPU_FP64, False, fgpu.FGPU_PC_NONE),
    (fgpu.FGPU_FP64, False, fgpu.FGPU_PC_CHEBYSHEV), (fgpu.FGPU_FP64, True, fgpu.FGPU_PC_JACOBI),
    (fgpu.FGPU_MIXED, False, fgpu.FGPU_PC_JACOBI), (fgpu.FGPU_MIXED, True, fgpu.FGPU_PC_JACOBI)])
@pytest.mark.parametrize("max_it, check_every", [(10000, 32), (37, 5), (1, 2)])
def test_folded_iterations_give_the_same_bits(ctx, small_mesh, precision, coarse, precond, max_it, check_every):
    tiny = M.make_tip_mesh(M.small_geometry(h_min=12.0, growth=0.8), with_atoms=False)
    # 8 cells per patch: about 2600 patches, above the limit, so no member of the batch folds
    big = _system(ctx, small_mesh, 8, coarse)
    assert big.mesh.patch_info()["n_patches"] > 2048
    # the Chebyshev degree of a batch follows its largest system
    o = fgpu.opts(tol=1e-10, max_it=max_it, check_every=check_every, precision=precision, precond=precond, inner_tol=0.01,
                  cheb_degree=4)
    out = []
    for others in ([], [big]):
        # a system of its own each time: Chebyshev keeps its estimate of the spectrum
        small = _system(ctx, tiny, 0, coarse)
        members = [small] + others
        for s in members:
            s.fill_solution(0.0)
        st = ctx.solve_batch(members, o)[0]
        out.append((st.iterations, st.outer, st.residual, small.solution()))
    assert out[0][:3] == out[1][:3]
    assert np.array_equal(out[0][3], out[1][3])
    assert (out[0][0] > 0) == (max_it == 10000)


@pytest.mark.parametrize("precision, precond", [(fgpu.FGPU_FP64, fgpu.FGPU_PC_JACOBI), (fgpu.FGPU_MIXED, fgpu.FGPU_PC_JACOBI),
                                                (fgpu.FGPU_FP64, fgpu.FGPU_PC_CHEBYSHEV)])
@pytest.mark.parametrize("terms", ["sigma", "heat"])
def test_folded_iterations_with_coefficients(ctx, small_mesh, precision, precond, terms):
    """The same for systems with coefficients per point: sigma(T), and kappa(T) with a mass term."""
    tiny = M.make_tip_mesh(M.small_geometry(h_min=12.0, growth=0.8), with_atoms=False)

    def system(tip, cells):
        gm = fgpu.Mesh(ctx, tip.nodes, tip.vacuum_cells(), *MARKS)
        if cells:
            gm.set_patch_cells(cells)
        xyz, _ = gm.dofs()
        cur, heat = fgpu.System(gm), fgpu.System(gm)
        heat.set_solution(300.0 + xyz[:, 2])
        if terms == "sigma":
            cur.reset()
            cur.sigma_terms(heat, 1.0, 3.9e-3)
            cur.add_dirichlet(2, 0.0)
            cur.add_neumann(8, None, -1.0)
            cur.apply_dirichlet()
            cur.fill_solution(0.0)
            return cur, heat
        cur.set_solution(0.01 * xyz[:, 0])
        heat.reset()
        heat.heat_terms(cur, serving.CU_RHO_CP / 4e-15, serving.LORENTZ)
        heat.add_dirichlet(2, 300.0)
        heat.apply_dirichlet()
        heat.fill_solution(300.0)
        return heat, cur

    o = fgpu.opts(tol=1e-10, precision=precision, precond=precond, inner_tol=0.01, cheb_degree=4)
    out = []
    for fold in (True, False):
        small = system(tiny, 0)
        members = [small] if fold else [small, system(small_mesh, 8)]
        assert fold or members[1][0].mesh.patch_info()["n_patches"] > 2048
        st = ctx.solve_batch([s for s, _ in members], o)[0]
        out.append((st.iterations, st.outer, st.residual, small[0].solution()))
    assert out[0][0] > 0 and out[0][:3] == out[1][:3]
    assert np.array_equal(out[0][3], out[1][3])
