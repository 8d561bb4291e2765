"""The ends of the multigrid hierarchy (a small level above a dense coarsest
in one workgroup; a dense coarsest alone on the grid; anything else through
the generic one-workgroup cycle) on meshes whose last levels differ, chosen by
the rows at which coarsening stops. The cycle is a fixed linear operator, so
beside the true residual each solve's iterations are compared with those the
generic cycle alone took on the same hierarchies, to one: two float32
summation orders may cross the tolerance one iteration apart."""

import numpy as np
import pytest

from bfm_amd import device as D
from bfm_amd import meshgen

pytestmark = pytest.mark.gpu


def solve(monkeypatch, nx, ny, kind, coarsest):
    monkeypatch.setenv("BFMX_AMG_COARSEST", str(coarsest))
    m = meshgen.beam(nx, ny, kind=kind, jitter=0.2, seed=4)
    s = D.beam_system(m)
    u, st = s.solve(precond=D.PRECOND_AMG, rtol=1e-9)
    A, b = s.get_csr_scipy(), s.get_rhs()
    assert st["status"] == 0
    assert np.linalg.norm(b - A @ u) <= 1.1e-9 * np.linalg.norm(b)
    return st["iterations"]


# iterations with coarsening down to 4, 16, 64 and 250 rows (250 on 153 nodes: the finest level dense)
EXPECTED = {
    (3, 16, 8): (31, 31, 29, 2), (3, 30, 20): (45, 39, 39, 36), (3, 64, 16): (24, 23, 23, 22),
    (3, 64, 35): (34, 34, 32, 32), (3, 120, 50): (38, 34, 34, 28), (3, 200, 100): (51, 41, 41, 31),
    (4, 16, 8): (28, 28, 26, 2), (4, 30, 20): (35, 33, 33, 32), (4, 64, 16): (18, 18, 18, 17),
    (4, 64, 35): (30, 29, 28, 28), (4, 120, 50): (24, 24, 24, 24), (4, 200, 100): (29, 29, 29, 29),
}


@pytest.mark.parametrize("kind,nx,ny", list(EXPECTED))
def test_ends_of_the_hierarchy(monkeypatch, kind, nx, ny):
    its = [solve(monkeypatch, nx, ny, kind, coarsest) for coarsest in (4, 16, 64, 250)]
    assert np.abs(np.subtract(its, EXPECTED[kind, nx, ny])).max() <= 1
