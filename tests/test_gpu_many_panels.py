"""Assembly of batches on either side of 1,024 systems (a launch a colour,
one workgroup a system): bitwise the same matrices and loads."""

import numpy as np
import pytest

from bfm_amd import device as D
from bfm_amd import meshgen

pytestmark = pytest.mark.gpu


def test_either_side_of_many():
    panels = [meshgen.panel(k, 400, 1000) for k in range(3)]
    inst = [D.panel_instance(*p) for p in panels]
    few = D.Batch.from_instances(inst)
    few.solve(rtol=1e-8)
    many = D.Batch.from_instances(inst * 342)   # 1,026
    many.solve(rtol=1e-8)
    for k in (0, 1, 2, 1023, 1024, 1025):
        a, b = few.system(k % 3), many.system(k)
        assert np.array_equal(a.get_rhs(), b.get_rhs())
        assert (a.get_csr_scipy() != b.get_csr_scipy()).nnz == 0
        assert np.array_equal(few.get_u(k % 3), many.get_u(k))
