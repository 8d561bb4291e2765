"""The learned preconditioner as a solve applies it, against the oracle, at
the edges of its 64-row tiles and on rows of different lengths (nodes of the
boundary and of P1 meshes). Six layers each split their input in two BF16
parts, a relative rounding of 2^-17 a layer; sums of mixed signs raise it by
up to some ten, hence 6 * 2^-17 * 10 = 5e-4, rounded up to 1e-3."""

import mpnn as M
import numpy as np
import pytest
from conftest import rel_err

from bfm_amd import device as D
from bfm_amd import meshgen

pytestmark = pytest.mark.gpu


# 4, 63, 64, 65, 128, 129 and 1,025 nodes
@pytest.mark.parametrize("kind", [3, 4])
@pytest.mark.parametrize("nx,ny", [(1, 1), (8, 6), (7, 7), (12, 4), (15, 7), (42, 2), (40, 24)])
def test_one_application(nx, ny, kind):
    mesh = meshgen.beam(nx, ny, kind=kind, jitter=0.2, seed=1)
    s = D.beam_system(mesh)
    fixed = np.zeros((mesh.n_nodes, 2), bool)
    fixed[s.node_perm()[np.asarray(mesh.node_sets["left"], bool)]] = True
    m = D.Model(seed=4)
    p = m.get_params()
    rng = np.random.default_rng(nx)
    p[M.OFF_W0:M.OFF_L] = 0.3 * rng.standard_normal(M.OFF_L - M.OFF_W0)
    m.set_params(p)
    s.set_model(m)
    G = M.Graph(*s.get_bsr(), M.features(*s.get_bsr(), fixed))
    r = rng.standard_normal((G.n, 2))
    r[fixed] = 0.0
    z = s.apply_model(r).reshape(-1, 2)
    y = G.block_jacobi(r)
    assert rel_err((z - y)[~fixed], (M.apply(p, G, r, bf=True) - y)[~fixed]) <= 1e-3
    s.set_model(None)
