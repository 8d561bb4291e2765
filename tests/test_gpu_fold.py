"""Flexible CG's coefficients from the partial sums its own kernels fold (up
to 1,024 workgroups of 256 rows) and from the reduction kernels (above): the
true residual is formed again from the matrix, and meshes on either side of
the line, which differ by one row of cells, take the same iterations to one."""

import numpy as np
import pytest

from bfm_amd import device as D
from bfm_amd import meshgen

pytestmark = pytest.mark.gpu


def solve(nx, ny):
    s = D.beam_system(meshgen.beam(nx, ny, kind=4, jitter=0.2, seed=6))
    u, st = s.solve(precond=D.PRECOND_AMG, rtol=1e-8)
    A, b = s.get_csr_scipy(), s.get_rhs()
    assert st["status"] == 0
    assert np.linalg.norm(b - A @ u) <= 1.1e-8 * np.linalg.norm(b)
    return st["iterations"]


# 255, 256, 258, 1,024 and 1,025 nodes; then 1,024 and 1,026 workgroups
@pytest.mark.parametrize("nx,ny", [(16, 14), (15, 15), (42, 5), (31, 31), (40, 24)])
def test_workgroups_of_the_partials(nx, ny):
    assert solve(nx, ny) > 0


def test_either_side_of_the_line():
    assert abs(solve(511, 511) - solve(511, 512)) <= 1
