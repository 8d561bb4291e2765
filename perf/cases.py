"""The work a user has this framework do, as cases that can be timed and checked.

Every case goes through a public entry point (the libbfm API by way of
bfm_amd.pybfm, or bfm_amd.device) and returns the whole result: displacements
in the mesh's own DOF order, or a training step's loss and gradient. The
ranges are those of the repository's workloads: 20% jittered beams from the
902-DOF one libbfm itself can solve to the 2,005,002-DOF one, holed panels of
1k-60k DOFs in batches, the learned preconditioner's training beams, and
axisymmetric rings.

kinds of case
    sim        pybfm Sim.run: host mesh in, displacements out (the drop-in)
    loads      a kept System, a new load vector, multigrid flexible CG
    design     a kept System, new element moduli: assemble, conditions, solve
    pcg        a kept System, its assembled load, Jacobi / block-Jacobi PCG
    batch_pcg  a kept Batch of holed panels: assembled and solved in one launch
    batch_amg  the same in the multigrid mode
    learned    flexible CG with the multigrid V-cycle and the network
    grad       loss and gradient of the network on recorded pairs
    axi        MINRES on an axisymmetric ring
"""

import math

import numpy as np
import torch

from bfm_amd import device as D
from bfm_amd import learned as L
from bfm_amd import meshgen
from bfm_amd import pybfm as pb

NU, RHO, STEEL = 0.3, 7850.0, 211e9
GRAVITY = (0.0, -9.81)


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the drop-in on the reference's own scale: every launch and copy counts
        dict(name="sim_902", kind="sim", nx=40, ny=10, el=3, stress=1),
        # the drop-in on a mesh libbfm's dense path can still hold
        dict(name="sim_10k", kind="sim", nx=121, ny=41, el=4, stress=1),
        # load cases on a small structure: latency of the multigrid solver
        dict(name="loads_2k", kind="loads", nx=64, ny=16, el=4),
        # load cases on the 2M-DOF beam: the bandwidth-bound end
        dict(name="loads_2m", kind="loads", nx=2000, ny=500, el=4),
        # a design loop: new moduli per element, assembled and solved again
        dict(name="design_502k", kind="design", nx=1000, ny=250, el=4, het=True),
        # the solver that System.solve takes by default, on a large system
        dict(name="pcg_502k", kind="pcg", nx=1000, ny=250, el=4, block=False, mixed=False),
        # mixed precision with block Jacobi, medium, heterogeneous triangles
        dict(name="mixed_46k", kind="pcg", nx=301, ny=75, el=3, block=True, mixed=True),
        # many small panels, one workgroup each
        dict(name="batch_pcg", kind="batch_pcg", count=256, hi=8000),
        # panels of the whole range as one multigrid system
        dict(name="batch_amg", kind="batch_amg", count=64, hi=60000),
        # the learned preconditioner on a held-out heterogeneous beam
        dict(name="learned_81k", kind="learned", nx=400, ny=100),
        # a training step's forward and backward pass
        dict(name="grad_13k", kind="grad", nx=160, ny=40, batch=8),
        # a ring, solved by MINRES
        dict(name="axi_902", kind="axi", nx=40, ny=10, el=4),
    ]


def _grid(rng, lo, hi):
    """Cells of a beam of about lo..hi DOFs (log-uniform), 3 to 5 times as long as high."""
    dofs = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    aspect = rng.uniform(3.0, 5.0)
    ny = max(4, int(round(math.sqrt(dofs / 2 / aspect))))
    return max(8, int(round(dofs / 2 / (ny + 1))) - 1), ny


def draw(rng):
    kind = rng.choice(("sim", "sim", "loads", "loads", "design", "design", "pcg", "pcg", "batch_pcg", "batch_amg",
                       "learned", "grad", "axi"))
    if kind == "sim":
        nx, ny = _grid(rng, 300, 12000)
        return dict(kind=kind, nx=nx, ny=ny, el=rng.choice((3, 4)), stress=rng.choice((0, 1)))
    if kind == "loads":
        nx, ny = _grid(rng, 1000, 1900000)
        return dict(kind=kind, nx=nx, ny=ny, el=rng.choice((3, 4)))
    if kind == "design":
        nx, ny = _grid(rng, 2000, 500000)
        return dict(kind=kind, nx=nx, ny=ny, el=rng.choice((3, 4)), het=rng.choice((True, False)))
    if kind == "pcg":
        mixed = rng.choice((True, False))
        nx, ny = _grid(rng, 1000, 46000 if mixed else 450000)
        return dict(kind=kind, nx=nx, ny=ny, el=rng.choice((3, 4)), block=rng.choice((True, False)), mixed=mixed)
    if kind == "batch_pcg":
        return dict(kind=kind, count=rng.randint(16, 250), hi=rng.randint(2000, 8000))
    if kind == "batch_amg":
        return dict(kind=kind, count=rng.randint(4, 64), hi=rng.randint(6000, 60000))
    if kind == "learned":
        nx, ny = _grid(rng, 2000, 80000)
        return dict(kind=kind, nx=nx, ny=ny)
    if kind == "grad":
        nx, ny = _grid(rng, 1000, 13000)
        return dict(kind=kind, nx=nx, ny=ny, batch=rng.randint(1, 8))
    nx, ny = _grid(rng, 200, 900)
    return dict(kind=kind, nx=nx, ny=ny, el=rng.choice((3, 4)))


# ----------------------------------------------------------------- the inputs

def _beam(case, seed):
    """The case's jittered beam, with moduli per element where it has them."""
    m = meshgen.beam(case["nx"], case["ny"], kind=case.get("el", 4), jitter=0.2, seed=seed)
    if case["kind"] == "learned" or (case["kind"] == "pcg" and case["mixed"]):
        m.elem_E = meshgen.loguniform_E(m.n_elems, seed=seed)
    if case["kind"] == "axi":
        m.coords = m.coords + np.array([1.0, 0.0])
    return m


def _traction(seed):
    return -1e6 * (0.5 + np.random.default_rng(seed).random())


def _load(mesh, seed):
    """A load case: a smooth pressure over the top edge, as nodal forces; nothing on the clamped edge."""
    rng = np.random.default_rng(seed + 31)
    amp = rng.normal(size=(2, 6)) * 1e6
    b = np.zeros((mesh.n_nodes, 2))
    e = mesh.edges.astype(np.int64)
    e = e[mesh.node_sets["top"][e].all(axis=1)]
    half = 0.5 * np.linalg.norm(mesh.coords[e[:, 0]] - mesh.coords[e[:, 1]], axis=1)
    for k in (0, 1):
        p = sum(amp[k, j] * np.cos(j * np.pi * mesh.coords[e[:, 0], 0] / 4.0) for j in range(6))
        np.add.at(b[:, k], e[:, 0], half * p)
        np.add.at(b[:, k], e[:, 1], half * p)
    b[mesh.node_sets["left"]] = 0.0
    return b.reshape(-1)


def _moduli(mesh, case, seed):
    """Element moduli of a design: log-uniform over two decades, or one modulus."""
    if case["het"]:
        return meshgen.loguniform_E(mesh.n_elems, seed=seed)
    return np.full(mesh.n_elems, STEEL * (0.5 + np.random.default_rng(seed).random()))


def _panels(case, seed):
    """The case's panels: their shapes are the case's, each one's traction and modulus the seed's."""
    rng = np.random.default_rng(seed + 47)
    out = []
    for k in range(case["count"]):
        mesh, t = meshgen.panel(k, 1000, case["hi"])
        out.append((mesh, t * (0.5 + rng.random()), dict(meshgen.PANEL_MATERIAL, E=STEEL * (0.5 + rng.random()))))
    return out


def _ring_conditions(mesh):
    s = mesh.node_sets
    return [1, 0, 3], [0.0, 0.0, -1e6], np.stack([s["bottom"], s["left"], s["top"]]).astype(np.uint8)


def _training_params():
    return L.default_params()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sim":
        mesh = _beam(case, seed)
        lib = pb.Library()
        cm = pb.Mesh_arrays.from_generated(mesh, lib=lib)
        obj = pb.Obj(cm, pb.Material("steel", RHO, STEEL, NU, lib=lib), pb.Rule_gauss_legendre(2, case["el"], lib=lib),
                     lib=lib)
        inst = pb.Instance(obj, lib=lib)
        keep = []
        for k, v, f in zip(*meshgen.beam_conditions(mesh, _traction(seed))):
            c = pb.Condition(cm, int(k), float(v), lib=lib)
            c.set_nodes(f)
            inst.add_condition(c)
            keep.append(c)
        sim = pb.Sim(pb.Sim.PLANAR_STRESS if case["stress"] else pb.Sim.PLANAR_STRAIN, lib=lib)
        sim.add_instance(inst)
        force = pb.Force_linear(GRAVITY, lib=lib)
        sim.add_force(force)
        return dict(kind=kind, sim=sim, inst=inst, keep=(cm, obj, keep, force))
    if kind == "loads":
        mesh = _beam(case, seed)
        return dict(kind=kind, s=D.beam_system(mesh), b=_load(mesh, seed))
    if kind == "design":
        mesh = _beam(case, seed)
        return dict(kind=kind, s=D.System.from_mesh(mesh), E=_moduli(mesh, case, seed),
                    conds=meshgen.beam_conditions(mesh, _traction(seed)))
    if kind == "pcg":
        mesh = _beam(case, seed)
        return dict(kind=kind, s=D.beam_system(mesh, traction=_traction(seed)),
                    precond=D.PRECOND_BLOCK_JACOBI if case["block"] else D.PRECOND_JACOBI,
                    precision=D.MIXED if case["mixed"] else D.FP64)
    if kind in ("batch_pcg", "batch_amg"):
        b = D.Batch.from_instances([D.panel_instance(m, t, mat) for m, t, mat in _panels(case, seed)])
        return dict(kind=kind, b=b, count=case["count"],
                    precond=D.PRECOND_BLOCK_JACOBI if kind == "batch_pcg" else D.PRECOND_AMG)
    if kind == "learned":
        mesh = _beam(case, seed)
        s = D.beam_system(mesh, traction=_traction(seed))
        s.set_model(D.Model(params=_training_params()))
        return dict(kind=kind, s=s)
    if kind == "grad":
        ts, model, _ = _training(case, seed)
        return dict(kind=kind, ts=ts, model=model, batch=case["batch"])
    mesh = _beam(case, seed)
    s = D.System.from_mesh(mesh)
    s.assemble(D.AXISYMMETRIC, 2.0e11, NU, RHO, g=GRAVITY)
    s.apply_conditions(*_ring_conditions(mesh))
    return dict(kind="axi", s=s)


def _training(case, seed):
    s = D.beam_system(_beam(case, seed), traction=_traction(seed))
    ts = D.TrainSet()
    ts.add(s, max_pairs=8, every=16, rtol=1e-9)
    return ts, D.Model(params=_training_params()), s


# ---------------------------------------------------------------- one pass

def run(state):
    kind = state["kind"]
    if kind == "sim":
        state["sim"].run()
        return state["inst"].effects
    if kind == "loads":
        return state["s"].solve(b=state["b"], precond=D.PRECOND_AMG)[0]
    if kind == "design":
        s = state["s"]
        s.assemble(True, STEEL, NU, RHO, elem_E=state["E"])
        s.apply_conditions(*state["conds"])
        return s.solve(precond=D.PRECOND_AMG)[0]
    if kind == "pcg":
        return state["s"].solve(precond=state["precond"], precision=state["precision"])[0]
    if kind in ("batch_pcg", "batch_amg"):
        b = state["b"]
        b.solve(precond=state["precond"])
        return np.concatenate([b.get_u(k) for k in range(state["count"])])
    if kind == "learned":
        return state["s"].solve(precond=D.PRECOND_AMG_LEARNED)[0]
    if kind == "grad":
        loss, grad = state["model"].loss_grad(state["ts"], 0, 0, state["batch"])
        return {"loss": loss, "grad": grad}
    return state["s"].solve(precond=D.PRECOND_MINRES)[0]


# ------------------------------------------------------- work and tolerance

def _size(case):
    """(nodes, blocks of the matrix) of the case: on average for panels, whose sizes are drawn."""
    if "count" in case:
        n = case["count"] * (1000 + case["hi"]) / 4
        return n, 7 * n
    n = (case["nx"] + 1) * (case["ny"] + 1)
    return n, (9 if case.get("el", 4) == 4 else 7) * n


def work(case):
    """What any solver has to read and write once: the matrix (or the mesh it is assembled from), the load, the
    displacements; a multiply-add per matrix entry. An iterative solver reads the matrix many times over: that is
    the algorithm's cost, not the problem's."""
    n, nnzb = _size(case)
    if case["kind"] == "grad":
        rows = n * case["batch"]
        # per row and layer (128 x 64): forward of x and of g, adjoint, and for each of the two gradients the
        # weight's and the input's product; r and e read, the parameters read and their gradient written
        return {"bytes": rows * 16 + nnzb * 20 + 2 * 4 * (128 + 3 * 8192), "flops": rows * 3 * 7 * 2 * 128 * 64}
    mixed = case.get("mixed", False)
    return {"bytes": nnzb * (20 if mixed else 36) + 2 * n * 8 * 2, "flops": nnzb * 8}


def tolerance(case):
    """Displacements of two solvers that both meet the relative residual (1e-8; 1e-10 for sim) but stop at other
    iterates: each was seen up to 7e-10 off the exact ones, and the error just before the stop is some ten times
    that. The network's products take BF16 inputs: the gradient was seen 1.3e-3 off the exact one."""
    return {"rel": 5e-3 if case["kind"] == "grad" else 3e-8}


# --------------------------------------------------------------- in 64 bits

_RULE = {3: ([1 / 6] * 3, [(1 / 6, 1 / 6), (1 - 1 / 3, 1 / 6), (1 / 6, 1 - 1 / 3)]),
         4: ([1.0] * 4, [(sx * 0.577350269189626, sy * 0.577350269189626)
                         for sx, sy in ((-1, 1), (-1, -1), (1, -1), (1, 1))])}


def _shape(el, x, y):
    if el == 3:
        return [1 - x - y, x, y], [-1, 1, 0], [-1, 0, 1]
    s = ((1, 1), (-1, 1), (-1, -1), (1, -1))
    return ([(1 + a * x) * (1 + b * y) / 4 for a, b in s], [a * (1 + b * y) / 4 for a, b in s],
            [b * (1 + a * x) / 4 for a, b in s])


def _elements(mesh, form, E, g):
    """Element matrices (elements, 2k, 2k) and the body load of the formulation (0 plane strain, 1 plane stress, 2
    axisymmetric, whose coefficients are those of the framework's documented formulas)."""
    el = mesh.kind
    nodes = mesh.elems.astype(np.int64)
    xy = mesh.coords[nodes]
    E = np.broadcast_to(np.asarray(E, np.float64), (len(nodes),))
    if form == 1:
        a, b = E / (1 - NU * NU), E * NU / (1 - NU * NU)
    else:
        a, b = E * (1 - NU) / (1 + NU) / (1 - 2 * NU), E * NU / (1 + NU) / (1 - 2 * NU)
    if form == 2:
        a = E * (1 - NU) / (1 + NU) * (1 - 2 * NU)
    c = E / (2 * (1 + NU))
    K = np.zeros((len(nodes), 2 * el, 2 * el))
    load = np.zeros((mesh.n_nodes, 2))
    for w, (px, py) in zip(*_RULE[el]):
        phi, dx, dy = (np.asarray(v, np.float64) for v in _shape(el, px, py))
        xx, xe, yx, ye = xy[:, :, 0] @ dx, xy[:, :, 0] @ dy, xy[:, :, 1] @ dx, xy[:, :, 1] @ dy
        det = np.abs(xx * ye - xe * yx)
        gx = (dx[None] * ye[:, None] - dy[None] * yx[:, None]) / det[:, None]
        gy = (dy[None] * xx[:, None] - dx[None] * xe[:, None]) / det[:, None]
        r = xy[:, :, 0] @ phi if form == 2 else np.ones(len(nodes))
        for j in range(el):
            for k in range(el):
                f11 = (a * gx[:, j] * gx[:, k] + c * gy[:, j] * gy[:, k]) * r
                f12 = (b * gx[:, j] * gy[:, k] + c * gy[:, j] * gx[:, k]) * r
                f21 = (b * gy[:, j] * gx[:, k] + c * gx[:, j] * gy[:, k]) * r
                f22 = a * gy[:, j] * gy[:, k] * r + c * gx[:, j] * gx[:, k]
                if form == 2:
                    f11 = f11 + phi[j] * (b * gx[:, k] + a * phi[k] / r) + gx[:, j] * b * phi[k]
                    f12 = f12 + phi[j] * b * gy[:, k]
                    f21 = f21 + gy[:, j] * b * phi[k]
                f = det * w
                K[:, 2 * j, 2 * k] += f * f11
                K[:, 2 * j, 2 * k + 1] += f * f12
                K[:, 2 * j + 1, 2 * k] += f * f21
                K[:, 2 * j + 1, 2 * k + 1] += f * f22
            if g is not None:
                np.add.at(load, nodes[:, j], (det * w * RHO * phi[j] * r)[:, None] * np.asarray(g)[None])
    return K, load


def _add_edge_load(mesh, load, flags, value, form):
    e = mesh.edges.astype(np.int64)
    e = e[flags.astype(bool)[e].all(axis=1)]
    p, q = mesh.coords[e[:, 0]], mesh.coords[e[:, 1]]
    f = 0.5 * np.linalg.norm(p - q, axis=1) * value
    if form == 2:
        s = 1 / math.sqrt(3)
        f = f * (p @ np.array([(1 - s) / 2, (1 + s) / 2]) + q @ np.array([(1 - s) / 2, (1 + s) / 2]))
    np.add.at(load[:, 1], e[:, 0], f)
    np.add.at(load[:, 1], e[:, 1], f)


def _direct(mesh, form, E, conds, g=None, b=None):
    """Displacements by block elimination over the mesh's columns of nodes, then refined with residuals in extended
    precision. Neumann-y and zero Dirichlet conditions only."""
    K, load = _elements(mesh, form, E, g)
    fixed = np.zeros((mesh.n_nodes, 2), bool)
    for kind, value, flags in zip(*conds):
        if kind == 3:
            _add_edge_load(mesh, load, np.asarray(flags), value, form)
    for kind, value, flags in zip(*conds):
        if kind < 2:
            fixed[np.asarray(flags, bool), kind] = True
    if b is not None:
        load = b.reshape(-1, 2).copy()
    load[fixed] = 0.0
    nodes = mesh.elems.astype(np.int64)
    dof = np.stack([2 * nodes, 2 * nodes + 1], 2).reshape(len(nodes), -1)
    free = ~fixed.reshape(-1)
    K *= (free[dof][:, :, None] & free[dof][:, None, :])
    # a node's column and its place there: the grid the mesh was cut from
    if "pins" in mesh.node_sets:
        col = np.unique(mesh.coords[:, 0], return_inverse=True)[1]
        row = np.unique(mesh.coords[:, 1], return_inverse=True)[1]
    else:
        nxp = int(mesh.node_sets["bottom"].sum())
        col, row = np.arange(mesh.n_nodes) % nxp, np.arange(mesh.n_nodes) // nxp
    nc, m = int(col.max()) + 1, 2 * (int(row.max()) + 1)
    place = np.stack([2 * row, 2 * row + 1], 1).reshape(-1)
    dcol = np.repeat(col, 2)
    diag = np.zeros((nc, m, m))
    off = np.zeros((nc, m, m))   # off[c]: rows of column c, columns of c + 1
    I = np.repeat(dof, dof.shape[1], axis=1).reshape(-1)
    J = np.tile(dof, (1, dof.shape[1])).reshape(-1)
    v = K.reshape(-1)
    for want, to in ((0, diag), (1, off)):
        at = np.nonzero(dcol[J] - dcol[I] == want)[0]
        flat = (dcol[I[at]] * m + place[I[at]]) * m + place[J[at]]
        to += np.bincount(flat, weights=v[at], minlength=nc * m * m).reshape(nc, m, m)
    there = np.zeros((nc, m), bool)
    there[dcol[free], place[free]] = True
    c_, p_ = np.nonzero(~there)
    diag[c_, p_, p_] = 1.0
    diag, off = torch.from_numpy(diag), torch.from_numpy(off)
    lu, fill = [], []
    S = diag[0]
    for c in range(nc):
        lu.append(torch.linalg.lu_factor(S))
        if c + 1 < nc:
            fill.append(torch.linalg.lu_solve(*lu[c], off[c]))
            S = diag[c + 1] - off[c].T @ fill[c]

    def solve(r):
        y = torch.zeros(nc, m, dtype=torch.float64)
        y[dcol, place] = torch.from_numpy(r)
        y = list(y.unsqueeze(-1))
        for c in range(nc):
            y[c] = torch.linalg.lu_solve(*lu[c], y[c])
            if c + 1 < nc:
                y[c + 1] = y[c + 1] - off[c].T @ y[c]
        for c in range(nc - 2, -1, -1):
            y[c] = y[c] - fill[c] @ y[c + 1]
        return torch.stack(y)[dcol, place, 0].numpy()

    load = load.reshape(-1)
    u = solve(load).astype(np.longdouble)
    Kl = K.astype(np.longdouble)
    for _ in range(2):
        part = np.matmul(Kl, u[dof][:, :, None])[:, :, 0]
        r = load.astype(np.longdouble)
        np.subtract.at(r, dof.reshape(-1), part.reshape(-1))
        r[~free] = 0
        u = u + solve(r.astype(np.float64))
    return u.astype(np.float64)


def _network(case, seed):
    """Loss and gradient of the network on the recorded pairs, in torch: z = D^-1 r + P S N^T N S P r with N three
    linear message-passing layers, loss the mean of (z - e)^T A (z - e) / (e^T A e)."""
    ts, model, s = _training(case, seed)
    rowptr, col, val = s.get_bsr()
    _, r, e, _, den = ts.get(0)
    mesh = _beam(case, seed)
    perm = s.node_perm()
    fixed = np.zeros(mesh.n_nodes, bool)
    fixed[perm[mesh.node_sets["left"]]] = True
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t = lambda x, k=torch.float64: torch.as_tensor(np.asarray(x), device=dev).to(k)  # noqa: E731
    n, B = mesh.n_nodes, case["batch"]
    r, e, den, A = t(r[:B]), t(e[:B]), t(den[:B]), t(val)
    I = t(np.repeat(np.arange(n), np.diff(rowptr)), torch.int64)
    J = t(col, torch.int64)
    diag = A[I == J]
    dinv = torch.linalg.inv(diag)
    scale = (0.5 * (diag[:, 0, 0] + diag[:, 1, 1])).rsqrt()
    keep = (~t(fixed, torch.bool)).to(torch.float64)[:, None] * scale[:, None]
    a = A * (scale[I] * scale[J])[:, None, None]
    w = a.reshape(-1, 4).repeat_interleave(16, dim=1)                       # weight per channel, entry (i, j)
    wt = a.transpose(1, 2).reshape(-1, 4).repeat_interleave(16, dim=1)      # of block (j, i), A symmetric
    p = t(model.get_params()).requires_grad_(True)
    W0 = p[:128].reshape(2, 64)
    Ws = [p[128 + 8192 * k:128 + 8192 * (k + 1)].reshape(128, 64) for k in range(3)]

    def gather(h, weight):
        return torch.stack([torch.zeros(n, 64, dtype=h.dtype, device=dev).index_add(0, I, weight * x[J]) for x in h])

    h = (r * keep) @ W0
    for W in Ws:
        h = torch.cat([h, gather(h, w)], -1) @ W
    x = h
    for W in reversed(Ws):
        o = x @ W.T
        x = o[..., :64] + gather(o[..., 64:], wt)
    z = torch.einsum("nij,bnj->bni", dinv, r) + (x @ W0.T) * keep
    d = z - e
    Ad = torch.stack([torch.zeros_like(x).index_add(0, I, torch.einsum("kij,kj->ki", A, x[J])) for x in d])
    loss = ((d * Ad).sum((1, 2)) / den).mean()
    loss.backward()
    return {"loss": float(loss.detach()), "grad": p.grad.cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "grad":
        return _network(case, seed)
    if kind in ("batch_pcg", "batch_amg"):
        return np.concatenate([_direct(m, 0, mat["E"], meshgen.panel_conditions(m, t))
                               for m, t, mat in _panels(case, seed)])
    if case["ny"] > 300:
        return None   # the elimination would take a minute
    mesh = _beam(case, seed)
    if kind == "axi":
        return _direct(mesh, 2, 2.0e11, _ring_conditions(mesh), g=GRAVITY)
    if kind == "loads":
        return _direct(mesh, 1, STEEL, meshgen.beam_conditions(mesh), b=_load(mesh, seed))
    conds = meshgen.beam_conditions(mesh, _traction(seed))
    if kind == "sim":
        return _direct(mesh, case["stress"], STEEL, conds, g=GRAVITY)
    if kind == "design":
        return _direct(mesh, 1, _moduli(mesh, case, seed), conds)
    return _direct(mesh, 1, STEEL if mesh.elem_E is None else mesh.elem_E, conds)
