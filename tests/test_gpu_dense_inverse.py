"""The dense inverse of the multigrid's coarsest level at the edges of its
register tiles (48, 96 and 192 rows): a system of at most 64 nodes has that
one level, whose preconditioner is the FP32 application of the inverse, so
flexible CG ends after very few iterations with the direct solve's
displacements (to the residual tolerance times the condition number, about
1e-10 x 1e4)."""

import numpy as np
import pytest

from conftest import rel_err

from bfm_amd import device as D
from bfm_amd import meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(2, 1), (4, 1), (5, 3), (11, 1), (12, 1), (7, 5), (15, 2), (24, 1), (7, 7)])
def test_small_systems_are_solved_by_their_inverse(nx, ny):
    s = D.beam_system(meshgen.beam(nx, ny, kind=4, jitter=0.2, seed=nx))
    u, st = s.solve(precond=D.PRECOND_AMG, rtol=1e-10)
    ref = np.linalg.solve(s.get_dense(), s.get_rhs())
    print(f"{2 * s.n_nodes} DOFs: {st['iterations']} iterations, error {rel_err(u, ref):.1e}")
    assert st["status"] == 0 and st["iterations"] <= 4
    assert rel_err(u, ref) <= 1e-6


def test_batches_of_segments():
    """Coarsest segments of different sizes inverted in one launch."""
    inst, ref = [], []
    for nx, ny in [(4, 1), (12, 1), (24, 1), (7, 7)]:
        m = meshgen.beam(nx, ny, kind=4, jitter=0.2, seed=nx)
        inst.append(D.planar_instance(m, True, meshgen.BEAM_MATERIAL, *meshgen.beam_conditions(m)))
        s = D.beam_system(m)
        ref.append(np.linalg.solve(s.get_dense(), s.get_rhs()))
    b = D.Batch.from_instances(inst)
    st, _ = b.solve(precond=D.PRECOND_AMG, rtol=1e-10)
    for k in range(len(inst)):
        assert st[k]["status"] == 0 and rel_err(b.get_u(k), ref[k]) <= 1e-6, k
