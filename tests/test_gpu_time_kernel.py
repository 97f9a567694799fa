"""Timing a CG iteration's kernels between the steps of a running batch, or on a solved system,
leaves the solves as they are: bits and iterations of systems that were never timed."""
import numpy as np
import pytest

from femocs_amd import fgpu
from femocs_amd import mesh as M

pytestmark = pytest.mark.gpu
MARKS = (8, 2, 4, 2)


def _system(ctx, tip, coarse):
    s = fgpu.System(fgpu.Mesh(ctx, tip.nodes, tip.vacuum_cells(), *MARKS))
    s.reset()
    s.add_dirichlet(2, 0.0)
    s.add_neumann(8, None, -1.0)
    s.apply_dirichlet()
    s.fill_solution(0.0)
    if coarse:
        s.set_coarse(True)
    return s


@pytest.mark.parametrize("precision, coarse", [(fgpu.FGPU_FP64, False), (fgpu.FGPU_FP64, True), (fgpu.FGPU_MIXED, False),
                                               (fgpu.FGPU_MIXED, True)])
@pytest.mark.parametrize("members", [1, 2])
def test_timing_between_steps(ctx, small_mesh, precision, coarse, members):
    tips = [small_mesh, M.make_tip_mesh(M.small_geometry(h_min=12.0, growth=0.8), with_atoms=False)][:members]
    o = fgpu.opts(tol=1e-9, precision=precision, inner_tol=0.1, use_graph=False)
    ref = [_system(ctx, t, coarse) for t in tips]
    want = [s.solve(o).iterations for s in ref]
    assert min(want) > 0
    kernels = [0, 1, 3] + ([2] if coarse and precision == fgpu.FGPU_MIXED else [])
    systems = [_system(ctx, t, coarse) for t in tips]
    b = fgpu.Batch(ctx, o)
    for s in systems:
        b.add(s)
    stats = {}
    while len(stats) < members:
        if len(b) == members:
            assert min(b.time_kernel(k, reps=3) for k in kernels) > 0
        b.step(24)
        stats.update(b.retire())
    for s, r, it in zip(systems, ref, want):
        assert stats[s].iterations == it and np.array_equal(s.solution(), r.solution())
        assert min(s.time_kernel(k, precision, 3) for k in kernels) > 0
        assert np.array_equal(s.solution(), r.solution())
    if 2 not in kernels:
        with pytest.raises(fgpu.FgpuError):
            systems[0].time_kernel(2, precision, 3)
