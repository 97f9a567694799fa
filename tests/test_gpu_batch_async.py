"""A member that finished is retired while the next step, of which it is still a member, is in flight,
and solved again at once: in the same batch, in another one, or alone.  The new solve starts after
that step, so its result has the bits and iterations of a solve alone."""
import numpy as np
import pytest

from femocs_amd import fgpu
from femocs_amd import mesh as M

pytestmark = pytest.mark.gpu
MARKS = (8, 2, 4, 2)


def _system(ctx, tip):
    s = fgpu.System(fgpu.Mesh(ctx, tip.nodes, tip.vacuum_cells(), *MARKS))
    s.reset()
    s.add_dirichlet(2, 0.0)
    s.add_neumann(8, None, -1.0)
    s.apply_dirichlet()
    s.fill_solution(0.0)
    return s


@pytest.mark.parametrize("precision", [fgpu.FGPU_FP64, fgpu.FGPU_MIXED])
@pytest.mark.parametrize("again", ["same batch", "another batch", "alone"])
def test_solved_again_behind_the_step_in_flight(ctx, small_mesh, precision, again):
    tiny = M.make_tip_mesh(M.small_geometry(h_min=12.0, growth=0.8), with_atoms=False)
    o = fgpu.opts(tol=1e-9, precision=precision, inner_tol=0.1, use_graph=False)
    ref = _system(ctx, tiny)
    alone = ref.solve(o)
    assert alone.iterations > 0
    first, slow = _system(ctx, tiny), _system(ctx, small_mesh)
    batch = fgpu.Batch(ctx, o)
    batch.add(first)
    batch.add(slow)
    running = 2
    while running == 2:                        # the small system is done first
        batch.step_async(8)
        running = batch.wait()
    assert running == 1
    batch.step_async(2000)                     # both are members of this step
    assert [s for s, _ in batch.retire()] == [first]
    first.fill_solution(0.0)
    if again == "alone":
        st = first.solve(o)
    else:
        b = batch if again == "same batch" else fgpu.Batch(ctx, o)
        b.add(first)
        batch.wait()
        stats = {}
        while first not in stats:
            b.step(32)
            stats.update(b.retire())
        st = stats[first]
    assert st.iterations == alone.iterations and np.array_equal(first.solution(), ref.solution())
