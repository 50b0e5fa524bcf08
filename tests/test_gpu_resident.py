"""Resident solves (``efea_solve_resident``, GPU tests): every kernel variant
against the classic iteration on the same system, paused and continued solves
against whole ones bit for bit, and the ways out (a block that waits too long,
a zero right-hand side, NaN)."""

import ctypes as C

import numpy as np
import pytest
import torch

import easyfea_amd as ea
from easyfea_amd import Models, Simulations, _lib
from easyfea_amd import device as dv
from easyfea_amd import resident as R
from easyfea_amd.mesh import tetra4_box
from test_resident_plan import irregular

pytestmark = pytest.mark.gpu


def _system(mesh, dof_n, seed=0):
    """(A, b, x0, known): an elastic stiffness, or a reaction-diffusion matrix."""
    rng = np.random.default_rng(seed)
    if dof_n > 1:
        E = np.exp(rng.normal(0.0, 0.2, mesh.Ne))
        simu = Simulations.Elastic(mesh, Models.Elastic.Isotropic(mesh.dim, E=E, v=0.3))
        A = simu._device_K()
    else:
        simu = Simulations.Thermal(mesh, Models.Thermal(np.exp(rng.normal(0.0, 0.3, mesh.Ne)), 1.0))
        K, M = simu._device_KC()
        A = dv.DeviceCsr(K.pattern)
        A.combine([(1.0, K), (float(mesh.Nn) ** (2 / mesh.dim) / 50, M)])
    known = np.zeros(mesh.Nn * dof_n, dtype=np.uint8)
    side = np.nonzero(mesh.coord[:, 0] == 0)[0]
    known.reshape(-1, dof_n)[side] = 1
    x0 = np.zeros(mesh.Nn * dof_n)
    x0.reshape(-1, dof_n)[side] = rng.normal(size=(side.size, dof_n)) * 1e-3
    return A, dv.to_dev(rng.normal(size=x0.size)), dv.to_dev(x0), dv.to_dev(known)


def _run(A, b, x0, known, precond, pipelined):
    job = dv.SolveJob(A, b, x0.clone(), known, "fp64", 1e-12, 1e-10, precond=precond, pipelined=pipelined)
    return job, job.run(raise_on_fail=False)


def _close(x, y, known):
    assert torch.equal(x[known != 0], y[known != 0])
    return float(torch.linalg.vector_norm(x - y) / torch.linalg.vector_norm(y))


Q, T, H = ea.quad4_rectangle, ea.tri3_rectangle, ea.hexa8_box
CASES = [  # mesh, dof_n, preconditioner, (slots, passes)
    (lambda: Q(1, 1, 1, 1), 2, "bj", (4, 1)),
    (lambda: Q(4, 1, 60, 3), 2, "bj", (5, 1)),           # one block
    (lambda: Q(1, 1, 15, 15), 2, "bj", (5, 1)),          # 256 nodes: one full block
    (lambda: Q(1, 1, 32, 31), 2, "two-level", (5, 1)),
    (lambda: T(1, 1, 33, 47), 2, "two-level", (4, 1)),
    (lambda: T(1, 1, 290, 250), 2, "two-level", (4, 2)),
    (lambda: Q(1, 1, 290, 250), 2, "two-level", (5, 2)),
    (lambda: T(1, 1, 400, 420), 2, "bj", (4, 4)),
    (lambda: Q(1, 1, 400, 420), 2, "two-level", (5, 4)),
    (lambda: T(1, 1, 40, 30), 1, "bj", (7, 1)),
    (lambda: T(1, 1, 420, 400), 1, "bj", (7, 2)),
    (lambda: T(1, 1, 600, 600), 1, "bj", (7, 4)),
    (lambda: Q(1, 1, 350, 353), 1, "bj", (9, 1)),
    (lambda: Q(1, 1, 420, 400), 1, "bj", (9, 2)),
    (lambda: Q(1, 1, 700, 610), 1, "bj", (9, 4)),
    (lambda: Q(1, 1, 730, 720), 1, "bj", (9, 9)),
    (lambda: T(1, 1, 730, 720), 1, "bj", (7, 9)),
    (lambda: H(1, 1, 1, 7, 9, 8), 1, "bj", (28, 1)),
    (lambda: H(1, 1, 1, 55, 54, 53), 1, "bj", (28, 2)),
    (lambda: tetra4_box(1, 1, 1, 9, 9, 9), 1, "bj", (16, 1)),
    (lambda: tetra4_box(1, 1, 1, 54, 55, 53), 1, "bj", (16, 2)),
    (lambda: H(1, 1, 1, 5, 6, 4), 3, "bj", (7, 1)),
    (lambda: H(1, 1, 1, 20, 19, 21), 3, "two-level", (7, 1)),
    (lambda: H(1, 1, 1, 30, 31, 29), 3, "two-level", (7, 1)),
    (lambda: tetra4_box(1, 1, 1, 17, 18, 17), 3, "two-level", (4, 1)),
    (lambda: tetra4_box(1, 1, 1, 35, 34, 33), 3, "two-level", (4, 2)),
    (lambda: tetra4_box(1, 1, 1, 6, 5, 4), 3, "bj", (4, 1)),
    # Delaunay meshes: rows of up to 11 nodes in 2D, 27 in 3D
    (lambda: irregular(30, 2, 2), 2, "bj", (8, 1)),
    (lambda: irregular(30, 2, 2), 2, "two-level", (8, 1)),
    (lambda: irregular(262, 2), 2, "two-level", (8, 2)),
    (lambda: irregular(30, 2, 2), 1, "bj", (16, 1)),
    (lambda: irregular(9, 3), 1, "bj", (28, 1)),
    (lambda: irregular(9, 3), 3, "bj", (7, 1)),
    (lambda: irregular(17, 3), 3, "two-level", (7, 1)),
    (lambda: irregular(262, 2), 2, "bj", (8, 2)),
    (lambda: T(1, 1, 290, 250), 2, "bj", (4, 2)),
    (lambda: Q(1, 1, 290, 250), 2, "bj", (5, 2)),
    (lambda: Q(1, 1, 400, 420), 2, "bj", (5, 4)),
    (lambda: T(1, 1, 400, 420), 2, "two-level", (4, 4)),
    (lambda: tetra4_box(1, 1, 1, 35, 34, 33), 3, "bj", (4, 2)),
]


def test_every_variant_has_a_case():
    """Each of EFEA_RESIDENT, and with aggregates those of two and three DOFs."""
    shapes = {(d, p, R.shape(d, n, k)[1:]) for d in (1, 2, 3) for n in range(1, 30) for k in range(1, 10)
              for p in ("bj", "two-level")[:d] if R.shape(d, n, k)}
    assert shapes == {(d, p, v) for _, d, p, v in CASES}


@pytest.mark.parametrize("case", range(len(CASES)))
def test_resident_matches_classic(case):
    make, dof_n, precond, variant = CASES[case]
    A, b, x0, known = _system(make(), dof_n)
    job, info = _run(A, b, x0, known, precond, "auto")
    p = job.resident.plan
    print(f"{A.Nn} nodes: {p.nblk} blocks, {info.iterations} iterations", flush=True)
    assert (p.slots, p.passes) == variant
    assert info.status == 1 and info.resident and not info.fallback
    classic, ci = _run(A, b, x0, known, precond, False)
    assert not ci.resident and abs(info.iterations - ci.iterations) <= 2 + ci.iterations // 50
    # both stop at an estimated 1e-10 in the energy norm
    assert _close(job.x, classic.x, known) < 1e-8
    assert info.rel_residual < 10 * max(ci.rel_residual, 1e-12)
    again, ai = _run(A, b, x0, known, precond, "auto")
    assert torch.equal(again.x, job.x) and ai.iterations == info.iterations


@pytest.mark.parametrize("case", [2, 3, 6, 13, 15, 23, 26])
def test_paused_solve_continues_bit_for_bit(case):
    make, dof_n, precond, _ = CASES[case]
    A, b, x0, known = _system(make(), dof_n)
    whole, wi = _run(A, b, x0, known, precond, "auto")
    for expected in (1, 9, wi.iterations - 4, wi.iterations):
        job = dv.SolveJob(A, b, x0.clone(), known, "fp64", 1e-12, 1e-10, precond=precond,
                          expected_iterations=max(1, expected))
        pending = job.start()
        assert pending is not None and pending.entry == "resident"
        info = pending.finish()
        queued = dv.deferred_budget(max(1, expected), pending.kind)
        assert pending.resumed == (queued <= wi.iterations)  # the test that ends it follows the last one
        assert torch.equal(job.x, whole.x)
        assert (info.iterations, info.rel_residual, info.status) == (wi.iterations, wi.rel_residual, 1)


def test_continued_solve_does_not_depend_on_what_ran_between():
    """The 9-pass variant: between the start and the finish, a solve of NaN on
    a system that fills its blocks leaves NaN in the LDS of the CUs, at the
    positions where the continued solve's blocks hold no node as well."""
    A, b, x0, known = _system(Q(1, 1, 730, 720), 1)
    B, c, y0, knownB = _system(Q(1, 1, 683, 767), 1)  # 114 blocks of 4608 nodes
    whole, wi = _run(A, b, x0, known, "bj", "auto")
    p = whole.resident.plan
    assert (p.slots, p.passes) == (9, 9) and p.nblk * 4608 > A.Nn
    y0.fill_(float("nan"))  # the last product is that of x
    job = dv.SolveJob(A, b, x0.clone(), known, "fp64", 1e-12, 1e-10, precond="bj", expected_iterations=9)
    pending = job.start()
    _run(B, c, y0, knownB, "bj", "auto")
    assert B.pattern.resident().plan.nblk * 4608 == B.Nn
    info = pending.finish()
    assert pending.resumed and info.resident and not info.fallback
    assert torch.equal(job.x, whole.x) and info.iterations == wi.iterations


def test_a_block_that_waits_too_long_gives_up(monkeypatch):
    """A wait limit no exchange can meet: the solve fails, every wait ends, and
    the classic iteration redoes it from the same start."""
    A, b, x0, known = _system(Q(1, 1, 60, 60), 2)
    _, ci = _run(A, b, x0, known, "two-level", False)
    monkeypatch.setattr(dv, "RESIDENT_WAIT_MS", 1e-9)
    job, info = _run(A, b, x0, known, "two-level", "auto")
    assert info.status == 1 and info.fallback and not info.resident and info.iterations == ci.iterations
    assert job.pipeline_failure[0] == _lib.ERR_NOCONV and "waited" in job.pipeline_failure[1]
    monkeypatch.undo()
    _, info = _run(A, b, x0, known, "two-level", "auto")
    assert info.status == 1 and info.resident


def test_solves_given_up_in_a_row_pause_the_resident_route(monkeypatch):
    """Two given up: none tried for 2 s, then one, and while it fails 4 s."""
    A, b, x0, known = _system(Q(1, 1, 60, 60), 2)
    now = [100.0]
    pauses = dv.ResidentPauses()
    pauses.clock = lambda: now[0]
    monkeypatch.setattr(dv, "resident_pauses", pauses)

    def tried():
        job, info = _run(A, b, x0, known, "two-level", "auto")
        assert info.status == 1
        return info.fallback, info.resident

    waits = dv.RESIDENT_WAIT_MS
    monkeypatch.setattr(dv, "RESIDENT_WAIT_MS", 1e-9)
    assert [tried() for _ in range(4)] == [(True, False)] * 2 + [(False, False)] * 2
    now[0] += 2.5
    assert [tried() for _ in range(2)] == [(True, False), (False, False)]
    now[0] += 2.5
    assert tried() == (False, False)
    job = dv.SolveJob(A, b, x0.clone(), known, "fp64", 1e-12, 1e-10, precond="bj", expected_iterations=9)
    pending = job.start()  # the pipelined form
    assert pending is not None and pending.entry == "pcgp" and pending.finish().status == 1
    monkeypatch.setattr(dv, "RESIDENT_WAIT_MS", waits)
    now[0] += 2.5
    assert [tried() for _ in range(2)] == [(False, True)] * 2


@pytest.mark.parametrize("precond", ["bj", "two-level"])
def test_the_iteration_limit_ends_the_solve(precond):
    """It is not run again by the classic iteration, which ends at the same iterate."""
    A, b, x0, known = _system(Q(1, 1, 60, 60), 2)
    xs = []
    for pipelined in ("auto", False):
        job = dv.SolveJob(A, b, x0.clone(), known, "fp64", 1e-12, 1e-10, precond=precond, pipelined=pipelined,
                          maxit=32)
        info = job.run(raise_on_fail=False)
        assert (info.status, info.fallback, info.resident) == (0, False, pipelined == "auto")
        assert info.rel_residual > 1e-6
        xs.append((job.x, info.iterations))
    assert xs[0][1] == xs[1][1]
    assert _close(xs[0][0], xs[1][0], known) < 1e-10
    with pytest.raises(_lib.EfeaError, match="not converged"):
        dv.SolveJob(A, b, x0.clone(), known, "fp64", 1e-12, 1e-10, precond=precond, maxit=32).run()


@pytest.mark.parametrize("dof_n,precond", [(1, "bj"), (2, "two-level")])
def test_zero_and_non_finite_right_hand_sides(dof_n, precond):
    A, b, x0, known = _system(Q(1, 1, 40, 40), dof_n)
    zero = torch.zeros_like(b)
    job, info = _run(A, zero, torch.zeros_like(b), known, precond, "auto")
    assert info.status == 1 and info.iterations == 0 and not job.x.any()
    b[17 * dof_n] = float("nan")
    for pipelined in ("auto", False):
        _, info = _run(A, b, x0, known, precond, pipelined)
        assert info.status == 2


@pytest.mark.parametrize("cells", [(40, 40), (730, 720)])  # one pass, nine
def test_an_unknown_row_of_zeros(cells):
    """block Jacobi puts 1 in place of a zero diagonal: the row stays at its start."""
    A, b, x0, known = _system(Q(1, 1, *cells), 1)
    n = A.Nn // 2
    at = torch.nonzero(A.pattern.node_cols == n).flatten()
    A.values[at] = 0.0
    A.values[int(A.node_ptr[n]):int(A.node_ptr[n + 1])] = 0.0
    b[n], x0[n] = 0.0, 0.25
    assert not known[n]
    job, info = _run(A, b, x0, known, "bj", "auto")
    assert job.resident.plan.passes == (1 if cells[0] == 40 else 9)
    assert info.status == 1 and info.resident and not info.fallback
    classic, _ = _run(A, b, x0, known, "bj", False)
    assert float(job.x[n]) == float(classic.x[n]) == 0.25
    assert _close(job.x, classic.x, known) < 1e-8
    b[n] = 1.0  # no solution
    for pipelined in ("auto", False):
        job = dv.SolveJob(A, b, x0.clone(), known, "fp64", 1e-12, 1e-10, precond="bj", pipelined=pipelined, maxit=300)
        info = job.run(raise_on_fail=False)
        assert info.status != 1


def test_two_threads_on_their_own_streams():
    """Solves of two threads at once take the chip in turn, with the results of
    one after the other."""
    import threading

    systems = [_system(Q(1, 1, 90 + 7 * k, 80), 2, seed=k) for k in range(2)]
    want = [_run(*s, "two-level", "auto")[0].x for s in systems]
    got, errors = [[], []], []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(6):
                    job, info = _run(*systems[k], "two-level", "auto")
                    got[k].append((info.resident, job.x))
        except Exception as exc:  # shown by the assertion below
            errors.append(exc)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    for k in range(2):
        for resident, x in got[k]:
            assert resident and torch.equal(x, want[k])


@pytest.mark.parametrize("mode,entry", [("fp64", "resident"), ("mixed", "pcgp")])
def test_a_start_ends_its_thread_s_open_one(mode, entry, monkeypatch):
    """A solve left open with too few iterations queued, as by a load step that
    raised, then another one's start on the same thread: both end as whole
    solves do, and so does one finished by another thread."""
    import threading

    monkeypatch.setattr(dv, "MIXED_MIN_MATRIX_BYTES", 0)
    systems = [_system(Q(1, 1, 40 + k, 33), 1, seed=k) for k in range(2)]

    def job(k, expected):
        A, b, x0, known = systems[k]
        return dv.SolveJob(A, b, x0.clone(), known, mode, 1e-12, 1e-10, precond="bj", expected_iterations=expected)

    whole = [job(k, 60) for k in range(2)]
    want = [w.run() for w in whole]

    def check(k, j, info):
        assert info.status == 1 and not info.fallback and info.iterations == want[k].iterations > 20
        assert torch.equal(j.x, whole[k].x)

    jobs = [job(0, 3), job(1, 60)]
    ws = dv.Workspace()  # of both: the second, larger one takes another buffer
    first, second = [j.start(ws) for j in jobs]
    assert first.entry == second.entry == entry
    for p in (second, first):
        check(jobs.index(p.job), p.job, p.finish())
    assert first.resumed and first.finish() is first.finish()

    j = job(0, 60)
    pending = j.start()
    t = threading.Thread(target=pending.finish)
    t.start()
    t.join()
    assert pending.resumed
    check(0, j, pending.finish())


def test_a_thread_for_each_solve():
    """Short-lived threads (each takes its event over from one that has ended)."""
    import threading

    A, b, x0, known = _system(Q(1, 1, 60, 60), 2)
    want = _run(A, b, x0, known, "two-level", "auto")[0].x
    got = []

    def work():
        with torch.cuda.stream(streams[len(got) % 2]):
            job, info = _run(A, b, x0, known, "two-level", "auto")
            got.append(info.resident and not info.fallback and torch.equal(job.x, want))

    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(12):
        t = threading.Thread(target=work)
        t.start()
        t.join()
    assert got == [True] * 12


def test_streams_of_one_handle():
    """hipStreamPerThread names another stream in each thread: the solves of two
    threads on it still take the chip in turn."""
    import threading

    per_thread = 2
    jobs, want, failed = [], [], []
    for k in range(2):
        A, b, x0, known = _system(T(1, 1, 251, 240 + 3 * k), 2, seed=k)
        want.append(_run(A, b, x0, known, "two-level", "auto")[0].x)
        job = dv.SolveJob(A, b, x0.clone(), known, "fp64", 1e-12, 1e-10, precond="two-level")
        job._prepare()
        assert job.resident.plan.nblk > 128  # two do not fit the chip together
        jobs.append((job, x0, dv.Workspace()))

    def work(k):
        job, x0, ws = jobs[k]
        raw = (C.c_double * 4)()
        for _ in range(6):
            with torch.cuda.stream(torch.cuda.Stream()):
                job.x.copy_(x0)
                torch.cuda.current_stream().synchronize()
            if _lib.call("efea_solve_resident", *job._resident_args(ws, 0), per_thread, raw) or raw[3] != 1 \
                    or not torch.equal(job.x, want[k]):
                failed.append(k)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed


@pytest.mark.parametrize("precond", ["bj", "two-level"])
def test_a_grid_cap_keeps_the_launch_per_step_iteration(precond):
    A, b, x0, known = _system(Q(1, 1, 60, 60), 2)

    def run(max_blocks, pipelined):
        job = dv.SolveJob(A, b, x0.clone(), known, "fp64", 1e-12, 1e-10, precond=precond, max_blocks=max_blocks,
                          pipelined=pipelined)
        return job, job.run()

    job, info = run(3, "auto")
    assert info.status == 1 and not info.resident and not info.fallback
    if precond == "bj":  # the cap is part of the order of the sums
        assert torch.equal(job.x, run(3, False)[0].x)
    assert run(0, "auto")[1].resident


def test_refused_arguments():
    lib = _lib.load()
    fake, info = 0x1000, (C.c_double * 4)()
    plan = _lib.ResidentPlan(dof_n=2, slots=5, passes=1, nblk=4, max_halo=10, nex=10, rows=fake, lidx=fake,
                             halo_ptr=fake, halo_ex=fake, pub=fake, pub_ptr=fake, pub_pos=fake, self=fake)
    args = [100, fake, fake, None, fake, None, None, 0, fake, fake, fake, 1 << 30, 1e-12, 1e-9, 10, 0, 0.0, None]
    assert lib.efea_solve_resident(C.byref(plan), 0, *args[1:], info) == -1
    plan.slots = 6
    assert lib.efea_solve_resident(C.byref(plan), *args, info) == -1 and "no kernel" in _lib.last_error()
    plan.slots, plan.nblk = 5, 300
    assert lib.efea_solve_resident(C.byref(plan), *args, info) == -1
    plan.nblk, plan.max_halo = 4, 20000  # more LDS than a CU has
    assert lib.efea_resident_fits(C.byref(plan)) == 0
    plan.max_halo, args[11] = 10, 16
    assert lib.efea_solve_resident(C.byref(plan), *args, info) == -4
    assert R.shape(2, 9, 1) == (2, 5, 1)
