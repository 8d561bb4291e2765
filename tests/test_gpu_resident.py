"""Jacobi PCG with the matrix in registers (bfm_amd/csrc/hip/resident.hip)
against the streaming kernels (BFMX_RESIDENT=0), at the edges of its
workgroups and of what it takes. Both runs meet the same true residual rtol,
which bounds each solution's error in the A-norm; the displacements are
compared to 1e-6, a hundred times what was seen, and the residual of the
register-resident solution is formed again from the matrix."""

import threading
import time

import numpy as np
import pytest

import mpnn as M
from conftest import rel_err

from bfm_amd import device as D
from bfm_amd import meshgen

pytestmark = pytest.mark.gpu

RTOL = 1e-9


def strip(n, kind, het, seed=5, h=None):
    """A beam of exactly n nodes: a grid h nodes high, cut off along its last column."""
    h = h or (4 if n < 256 else 16 if n < 1000 else 32 if n < 4000 else 96)
    nx = -(-n // h)
    m = meshgen.beam(nx, h - 1, kind=kind, length=nx / h, height=1.0, jitter=0.2, seed=seed)
    # nodes column by column, so that the first n of them are a prefix of the grid
    j, i = np.divmod(np.arange(m.n_nodes), nx + 1)
    order = np.argsort(i * h + j, kind="stable")
    new = np.empty_like(order)
    new[order] = np.arange(order.size)
    elems = new[m.elems.astype(np.int64)]
    elems = elems[(elems < n).all(axis=1)]
    edges = new[m.edges.astype(np.int64)]
    edges = edges[(edges < n).all(axis=1)]
    used = np.zeros(n, bool)
    used[elems.ravel()] = True
    assert used.all()
    sets = {k: v[order][:n] for k, v in m.node_sets.items()}
    out = meshgen.Mesh(kind, m.coords[order][:n].copy(), elems.astype(np.uint64), edges.astype(np.uint64),
                       -np.ones(len(edges), np.int64), sets)
    if het:
        out.elem_E = meshgen.loguniform_E(out.n_elems, seed=seed)
    return out


def both(monkeypatch, s, **kw):
    monkeypatch.setenv("BFMX_RESIDENT", "0")
    ref, st_ref = s.solve(**kw)
    monkeypatch.delenv("BFMX_RESIDENT")
    u, st = s.solve(**kw)
    return ref, st_ref, u, st


def check(s, u, ref, st, rtol):
    assert st["status"] == 0 and st["rel_residual"] <= rtol
    A, b = s.get_csr_scipy(), s.get_rhs()
    assert np.linalg.norm(b - A @ u) <= 1.1 * rtol * np.linalg.norm(b)
    assert rel_err(u, ref) <= 1e-6


# one workgroup of 512 and of 1024 threads, then clusters: full, a few rows less and over, an uneven last one
@pytest.mark.parametrize("n", [8, 64, 511, 512, 514, 515, 1022, 1023, 1024, 1026, 1027, 2047, 2048, 2050, 2051, 3200])
@pytest.mark.parametrize("kind,pre,precision", [(4, D.PRECOND_JACOBI, D.FP64), (3, D.PRECOND_BLOCK_JACOBI, D.FP64),
                                                (4, D.PRECOND_BLOCK_JACOBI, D.MIXED)])
def test_workgroup_edges(monkeypatch, n, kind, pre, precision):
    if precision == D.MIXED and n < 500:
        pytest.skip("the FP32 operator stalls above rtol on the smallest strips, on either path")
    m = strip(n, kind, het=pre == D.PRECOND_BLOCK_JACOBI and precision == D.FP64)
    assert m.n_nodes == n
    s = D.beam_system(m)
    rtol = 1e-8 if precision == D.MIXED else RTOL
    ref, st_ref, u, st = both(monkeypatch, s, precond=pre, precision=precision, rtol=rtol)
    print(f"{m.n_nodes} nodes: {st_ref['iterations']} / {st['iterations']} iterations, difference {rel_err(u, ref):.1e}")
    check(s, u, ref, st, rtol)
    again, st2 = s.solve(precond=pre, precision=precision, rtol=rtol)
    assert np.array_equal(u, again) and st2["iterations"] == st["iterations"]


# Columns of 600 and 900 nodes in their own order: a workgroup of 1,024 rows reads some 1,200 and 1,800 nodes of
# others (more than one a thread; 2,826 is near the widest window), one of MINRES's 512 rows the same.
@pytest.mark.parametrize("n,h,pre,precision",
                         [(6000, 600, D.PRECOND_JACOBI, D.FP64), (6005, 600, D.PRECOND_BLOCK_JACOBI, D.FP64),
                          (6050, 600, D.PRECOND_JACOBI, D.MIXED), (7200, 900, D.PRECOND_BLOCK_JACOBI, D.FP64),
                          (6000, 600, D.PRECOND_MINRES, D.FP64)])
def test_wide_windows(monkeypatch, n, h, pre, precision):
    s = D.beam_system(strip(n, 4, het=False, h=h), renumber=False)
    kw = dict(precond=pre, precision=precision, rtol=1e-8, max_iter=20000)
    ref, st_ref, u, st = both(monkeypatch, s, **kw)
    print(f"{n} nodes: {st_ref['iterations']} / {st['iterations']} iterations, difference {rel_err(u, ref):.1e}")
    assert not np.array_equal(u, ref)        # it was not streamed
    check(s, u, ref, st, 1e-8)
    monkeypatch.setenv("BFMX_RESIDENT_ITERS", "48")
    u2, st2 = s.solve(**kw)
    assert st2["iterations"] == st["iterations"] and np.array_equal(u, u2)


@pytest.mark.parametrize("nx,ny", [(70, 20), (480, 69), (1200, 100)])
def test_minres_of_many_workgroups(monkeypatch, nx, ny):
    """Three, 66 and 237 workgroups of 512 rows (most with neighbours on both sides; the sums over more than 64 are
    gathered by several wavefronts). Both paths are cut after 100 iterations, before the Lanczos vectors lose their
    orthogonality: the same recurrences in another order of summation, whose iterates agree to 1e-10 (seen 1e-12)."""
    s = D.beam_system(meshgen.beam(nx, ny, kind=4, jitter=0.2, seed=3))

    def iterate():
        with pytest.raises(D.BfmxError) as e:
            s.solve(precond=D.PRECOND_MINRES, rtol=1e-10, max_iter=100)
        assert e.value.code == -5 and "100 iterations" in str(e.value)
        return s.get_u()

    monkeypatch.setenv("BFMX_RESIDENT", "0")
    ref = iterate()
    monkeypatch.delenv("BFMX_RESIDENT")
    u = iterate()
    print(f"{s.n_nodes} nodes: difference {rel_err(u, ref):.1e}")
    assert not np.array_equal(u, ref) and rel_err(u, ref) <= 1e-10
    monkeypatch.setenv("BFMX_RESIDENT_ITERS", "7")
    assert np.array_equal(iterate(), u)


@pytest.mark.parametrize("nx,ny,precision", [(24, 6, D.FP64), (80, 20, D.FP64), (80, 20, D.MIXED)])
def test_a_run_cut_into_launches_is_the_same_run(monkeypatch, nx, ny, precision):
    s = D.beam_system(meshgen.beam(nx, ny, kind=4, jitter=0.2, seed=3))
    u, st = s.solve(precision=precision, rtol=1e-8)
    monkeypatch.setenv("BFMX_RESIDENT_ITERS", "48")
    u2, st2 = s.solve(precision=precision, rtol=1e-8)
    assert st["iterations"] > 96 and st2["iterations"] == st["iterations"] and np.array_equal(u, u2)


def test_what_does_not_fit_takes_the_streaming_kernels(monkeypatch):
    # a fan: the middle node's row has 13 blocks, more than the registers hold
    k = 12
    a = 2 * np.pi * np.arange(k) / k
    coords = np.concatenate([[[0.0, 0.0]], np.stack([np.cos(a), np.sin(a)], 1)])
    elems = np.array([[0, 1 + i, 1 + (i + 1) % k] for i in range(k)], np.uint64)
    s = D.System(3, coords, elems)
    s.assemble(1, 2e11, 0.3, 7850.0, g=(0.0, -9.81))
    fix = np.zeros(k + 1, np.uint8)
    fix[1:4] = 1
    s.apply_conditions([0, 1], [0.0, 0.0], [fix, fix])
    ref, _, u, st = both(monkeypatch, s, rtol=RTOL)
    assert np.array_equal(u, ref)
    # an order of the nodes that reaches over more than a window holds
    m = meshgen.beam(120, 50, kind=4, jitter=0.2, seed=4)
    p = np.random.default_rng(1).permutation(m.n_nodes)
    q = np.empty_like(p)
    q[p] = np.arange(p.size)
    m.coords, m.elems, m.edges = m.coords[p], q[m.elems.astype(np.int64)].astype(np.uint64), q[m.edges.astype(np.int64)]
    m.node_sets = {name: v[p] for name, v in m.node_sets.items()}
    s = D.beam_system(m, renumber=False)
    ref, _, u, st = both(monkeypatch, s, rtol=RTOL)
    assert np.array_equal(u, ref)
    s = D.beam_system(m)                    # renumbered, it fits
    ref, _, u, st = both(monkeypatch, s, rtol=RTOL)
    check(s, u, ref, st, RTOL)


def test_zero_load_limit_and_floor():
    s = D.beam_system(meshgen.beam(80, 20, kind=4, jitter=0.2, seed=3))
    u, st = s.solve(b=np.zeros(2 * s.n_nodes))
    assert st["iterations"] == 0 and np.array_equal(u, np.zeros_like(u))
    with pytest.raises(D.BfmxError) as e:
        s.solve(max_iter=20)
    assert e.value.code == -5 and "32 iterations" in str(e.value)   # whole rounds of 16
    with pytest.raises(D.BfmxError) as e:
        s.solve(rtol=1e-17)
    assert e.value.code == -8
    u, st = s.solve(rtol=RTOL)
    u2, st2 = s.solve(rtol=RTOL, max_iter=2**63 - 1)   # as good as no limit
    assert st2["status"] == 0 and np.array_equal(u, u2)


def test_clusters_on_several_threads():
    """More workgroups than the GPU holds at once, from several threads: each system's run is its own."""
    systems = [D.beam_system(meshgen.beam(400 + 10 * k, 180, kind=4, jitter=0.2, seed=k)) for k in range(4)]
    alone = [s.solve(rtol=1e-6)[0] for s in systems]
    got = [None] * len(systems)

    def work(k):
        for _ in range(2):
            got[k] = systems[k].solve(rtol=1e-6)[0]

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(systems))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(np.array_equal(a, g) for a, g in zip(alone, got))


def test_clusters_beside_each_other():
    """Clusters of 2 to 59 workgroups from twelve threads and a batch: each run is its own, bitwise, so that no
    wait ran out."""
    systems = [D.beam_system(meshgen.beam(60 + 50 * k, 20 + 7 * k, kind=3 + k % 2, jitter=0.2, seed=k))
               for k in range(12)]
    alone = [s.solve(rtol=1e-5)[0] for s in systems]
    batch = D.Batch(systems[::4])
    batch.solve(rtol=1e-5)
    in_batch = [batch.get_u(k) for k in range(3)]
    wrong = []

    def work(k):
        for _ in range(6):
            if k == 12:
                batch.solve(rtol=1e-5)
                ok = all(np.array_equal(batch.get_u(j), in_batch[j]) for j in range(3))
            else:
                ok = np.array_equal(systems[k].solve(rtol=1e-5)[0], alone[k])
            if not ok:
                wrong.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(13)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_a_small_solve_does_not_wait_for_a_large_one():
    """5,124 nodes (six workgroups) beside a thread that solves 201,051 nodes (197) over and over: on average well
    under the time of a large solve (4 of 38 ms seen, 39 when clusters ran one at a time)."""
    large = D.beam_system(meshgen.beam(800, 250, kind=4, jitter=0.2, seed=1))
    small = D.beam_system(meshgen.beam(182, 27, kind=4, jitter=0.2, seed=2))
    want, _ = small.solve(rtol=1e-6)
    large.solve(rtol=1e-4)
    t = time.perf_counter()
    large.solve(rtol=1e-4)
    t_large = time.perf_counter() - t
    stop = threading.Event()

    def work():
        while not stop.is_set():
            large.solve(rtol=1e-4)

    thread = threading.Thread(target=work)
    thread.start()
    time.sleep(0.5 * t_large)
    t = time.perf_counter()
    got = [small.solve(rtol=1e-6)[0] for _ in range(10)]
    t_small = (time.perf_counter() - t) / 10
    stop.set()
    thread.join()
    print(f"large {t_large * 1e3:.1f} ms, small beside it {t_small * 1e3:.1f} ms")
    assert all(np.array_equal(u, want) for u in got)
    assert t_small < 0.5 * t_large


@pytest.mark.parametrize("pre", [D.PRECOND_JACOBI, D.PRECOND_BLOCK_JACOBI])
def test_batches_of_clusters(monkeypatch, pre):
    """Clusters of many sizes in one batch, Q1 and P1, with a system that does not fit (it takes the streaming
    kernel in the same call); each against the streaming kernel and, bitwise, a batch of its own."""
    systems = [D.beam_system(strip(n, 3 + k % 2, het=False, seed=k))
               for k, n in enumerate((64, 1024, 1026, 2050, 3200, 5000, 7000, 9000, 12500, 20600, 2048, 30002))]
    wide = meshgen.beam(120, 50, kind=4, jitter=0.2, seed=4)
    p = np.random.default_rng(1).permutation(wide.n_nodes)
    q = np.empty_like(p)
    q[p] = np.arange(p.size)
    wide.coords, wide.elems = wide.coords[p], q[wide.elems.astype(np.int64)].astype(np.uint64)
    wide.edges = q[wide.edges.astype(np.int64)]
    wide.node_sets = {name: v[p] for name, v in wide.node_sets.items()}
    systems.insert(5, D.beam_system(wide, renumber=False))
    b = D.Batch(systems)
    monkeypatch.setenv("BFMX_RESIDENT", "0")
    st_ref, _ = b.solve(precond=pre, rtol=1e-8)
    ref = [b.get_u(k) for k in range(len(systems))]
    monkeypatch.delenv("BFMX_RESIDENT")
    st, _ = b.solve(precond=pre, rtol=1e-8)
    for k, s in enumerate(systems):
        assert st[k]["status"] == 0 and st[k]["rel_residual"] <= 1e-8, k
        u = b.get_u(k)
        assert rel_err(u, ref[k]) <= 1e-6, k
        A, f = s.get_csr_scipy(), s.get_rhs()
        assert np.linalg.norm(f - A @ u) <= 1.1e-8 * np.linalg.norm(f), k
        one = D.Batch([s])
        one.solve(precond=pre, rtol=1e-8)
        assert np.array_equal(one.get_u(0), u), k


@pytest.mark.parametrize("pre", [D.PRECOND_JACOBI, D.PRECOND_BLOCK_JACOBI])
def test_a_system_after_a_broken_one(pre):
    """A cluster's size is rounded up: 28,700 and 29,000 nodes leave two and one of its 32 workgroups without rows.
    They follow systems of NaN moduli on the same clusters (eight of 32 workgroups fill the GPU), whose NaNs stay
    behind in the workgroups' memory; their runs are those of a batch without the broken ones."""
    wide = strip(32000, 3, het=False)
    bad = [D.beam_system(wide, material=dict(meshgen.BEAM_MATERIAL, E=float("nan"))) for _ in range(8)]
    good = [D.beam_system(strip(n, 3, het=False)) for n in (29000, 28700)]
    alone = D.Batch(good)
    alone.solve(precond=pre, rtol=1e-6)
    b = D.Batch(bad + good)
    st, _ = b.solve(precond=pre, rtol=1e-6, check=False)
    assert all(x["status"] == -4 for x in st[:8])
    for k in range(2):
        assert st[8 + k]["status"] == 0
        assert np.array_equal(b.get_u(8 + k), alone.get_u(k))


def test_autotune_times_what_streams(monkeypatch):
    """Configurations apply to the systems that fit no cluster; only these are timed, each in its size class."""
    fit = [D.beam_system(strip(n, 4, het=False)) for n in (200, 3000, 9000)]
    wide = meshgen.beam(120, 50, kind=4, jitter=0.2, seed=4)     # 6,171 nodes in no order: the middle class
    p = np.random.default_rng(1).permutation(wide.n_nodes)
    q = np.empty_like(p)
    q[p] = np.arange(p.size)
    wide.coords, wide.elems = wide.coords[p], q[wide.elems.astype(np.int64)].astype(np.uint64)
    wide.edges = q[wide.edges.astype(np.int64)]
    wide.node_sets = {name: v[p] for name, v in wide.node_sets.items()}
    streams = D.beam_system(wide, renumber=False)
    b = D.Batch(fit)
    default, times = b.autotune(iters=8)
    assert not times.any()
    u = [b.solve(rtol=1e-6, picks=default) and b.get_u(k) for k in range(3)]
    picks, times = D.Batch([fit[2], streams, fit[0], fit[1]]).autotune(iters=8)
    assert (times[1] > 0).all() and not times[0].any() and not times[2].any()
    assert picks[1] == times[1].argmin() and picks[0] == default[0] and picks[2] == default[2]
    monkeypatch.setenv("BFMX_RESIDENT", "0")
    _, times = b.autotune(iters=8)
    assert (times > 0).all()
    monkeypatch.delenv("BFMX_RESIDENT")
    b.solve(rtol=1e-6)
    assert all(np.array_equal(b.get_u(k), u[k]) for k in range(3))


def ring(nx, ny, kind=4):
    """An axisymmetric ring (indefinite: MINRES)."""
    m = meshgen.beam(nx, ny, kind=kind, length=4.0, height=1.0, jitter=0.2, seed=12)
    m.coords = m.coords + np.array([1.0, 0.0])
    s = D.System.from_mesh(m)
    s.assemble(D.AXISYMMETRIC, 2.0e11, 0.3, 7850.0, g=(0.0, -9.81))
    sets = m.node_sets
    s.apply_conditions([1, 0, 3], [0.0, 0.0, -1e6], [sets["bottom"], sets["left"], sets["top"]])
    return s


# A wait that runs out is forced by a limit of one poll: every workgroup still ends, some of them on sums to which a
# failed one contributed. What comes back is bitwise the streaming kernels' solution and report. It costs seconds with
# the ordinary limit, so the system's or batch's next solve streams without trying; a new one is not held up.

@pytest.mark.parametrize("pre,precision,nx", [(D.PRECOND_JACOBI, D.FP64, 80), (D.PRECOND_BLOCK_JACOBI, D.FP64, 500),
                                              (D.PRECOND_JACOBI, D.MIXED, 120), (D.PRECOND_MINRES, D.FP64, 60)])
def test_a_wait_that_runs_out(monkeypatch, pre, precision, nx):
    s = ring(nx, 14) if pre == D.PRECOND_MINRES else D.beam_system(meshgen.beam(nx, 20, kind=4, jitter=0.2, seed=3))
    kw = dict(precond=pre, precision=precision, rtol=1e-7)
    ref, st_ref, u, st = both(monkeypatch, s, **kw)
    assert not np.array_equal(u, ref)          # the two paths differ in rounding
    monkeypatch.setenv("BFMX_RESIDENT_POLLS", "1")
    got, st_got = s.solve(**kw)
    assert np.array_equal(got, ref)
    assert [st_got[k] for k in ("status", "iterations", "rel_residual", "restarts")] == \
        [st_ref[k] for k in ("status", "iterations", "rel_residual", "restarts")]
    monkeypatch.delenv("BFMX_RESIDENT_POLLS")
    assert np.array_equal(s.solve(**kw)[0], ref)


def test_a_wait_that_runs_out_in_a_warm_start(monkeypatch):
    """The learned solve's block-Jacobi run from the iterate where a network that returns NaN broke down."""
    s = D.beam_system(meshgen.beam(80, 20, kind=4, jitter=0.2, seed=3))
    m = D.Model(seed=5)
    p = m.get_params()
    p[M.OFF_W0 + 3] = np.nan
    m.set_params(p)
    s.set_model(m)
    kw = dict(precond=D.PRECOND_LEARNED, rtol=1e-7)
    ref, st_ref, u, st = both(monkeypatch, s, **kw)
    assert st["fallback"] == 1 and not np.array_equal(u, ref)
    monkeypatch.setenv("BFMX_RESIDENT_POLLS", "1")
    got, st_got = s.solve(**kw)
    assert np.array_equal(got, ref) and st_got["iterations"] == st_ref["iterations"]


def test_a_wait_that_runs_out_in_a_batch(monkeypatch):
    systems = [D.beam_system(strip(n, 3 + k % 2, het=False, seed=k))
               for k, n in enumerate((64, 1026, 2050, 5000, 5100, 9000, 20600, 30002, 30002))]
    b = D.Batch(systems)
    monkeypatch.setenv("BFMX_RESIDENT", "0")
    st_ref, _ = b.solve(rtol=1e-6)
    ref = [b.get_u(k) for k in range(len(systems))]
    monkeypatch.delenv("BFMX_RESIDENT")
    monkeypatch.setenv("BFMX_RESIDENT_POLLS", "1")
    st, _ = b.solve(rtol=1e-6)
    for k in range(len(systems)):
        assert [st[k][x] for x in ("status", "iterations", "rel_residual")] == \
            [st_ref[k][x] for x in ("status", "iterations", "rel_residual")], k
        assert np.array_equal(b.get_u(k), ref[k]), k
    monkeypatch.delenv("BFMX_RESIDENT_POLLS")
    b.solve(rtol=1e-6)
    assert all(np.array_equal(b.get_u(k), ref[k]) for k in range(len(systems)))
    fresh = D.Batch(systems)
    fresh.solve(rtol=1e-6)
    assert not all(np.array_equal(fresh.get_u(k), ref[k]) for k in range(len(systems)))


@pytest.mark.parametrize("nx,ny,kind", [(3, 2, 3), (16, 5, 4), (40, 10, 4), (42, 11, 3), (51, 9, 4), (60, 14, 4)])
def test_minres(monkeypatch, nx, ny, kind):
    """Axisymmetric rings of 12 to 915 nodes (one workgroup of 512, and two) against the recurrences on the host;
    a run cut into launches is the same run. K is indefinite with a condition number of about 1e5 here: two
    solutions whose residuals meet 1e-8 agree to 1e-3 at the worst; seen 2e-9, of which a hundred times is allowed."""
    s = ring(nx, ny, kind)
    kw = dict(precond=D.PRECOND_MINRES, rtol=1e-8)
    ref, st_ref, u, st = both(monkeypatch, s, **kw)
    print(f"{s.n_nodes} nodes: {st_ref['iterations']} / {st['iterations']} iterations, difference {rel_err(u, ref):.1e}")
    assert abs(st["iterations"] - st_ref["iterations"]) <= 0.1 * st_ref["iterations"] + 10
    A, b = s.get_csr_scipy(), s.get_rhs()
    assert st["status"] == 0 and np.linalg.norm(b - A @ u) <= 1.1e-8 * np.linalg.norm(b)
    assert rel_err(u, ref) <= 2e-7
    monkeypatch.setenv("BFMX_RESIDENT_ITERS", "7")
    u2, st2 = s.solve(**kw)
    assert st2["iterations"] == st["iterations"] and np.array_equal(u, u2)
    monkeypatch.delenv("BFMX_RESIDENT_ITERS")
    u0, st0 = s.solve(b=np.zeros(2 * s.n_nodes), **kw)
    assert st0["iterations"] == 0 and not u0.any()
    with pytest.raises(D.BfmxError) as e:
        s.solve(precond=D.PRECOND_MINRES, rtol=1e-8, max_iter=5)
    assert e.value.code == -5 and "5 iterations" in str(e.value)
