"""Which launches a solve takes: resident ones where the system fits the chip,
the launch per phase where it does not or where a resident launch had to leave.
The counts of the system's resident batches tell them apart, so that a solve
that quietly took the other way does not pass for one that was tested."""
import time

import numpy as np
import pytest

import ogs5_amd as ox
from ogs5_amd import workloads as W

from test_gpu_resident import _same, _scenario, _solve

pytestmark = pytest.mark.gpu


def test_one_workgroup_launches_keep_out_of_the_census_ring():
    """The census entries of a system's launches are used again after 64 of
    them, and cleared by the launches half a ring before.  A launch of one
    workgroup clears none, so it may not be numbered among them: here a launch
    that left (decision 2) is followed by 40 launches of one workgroup and then
    by more than a ring of counted ones, none of which may find its entry with
    the old decision and leave."""
    sc = _scenario("quad", (40, 40))  # CG: one workgroup; BiCGStab: several
    system = W.make_system(sc, ox.FP64)
    s = system[1]
    s.resident_fail(ox.RESIDENT_LEAVE)
    _solve(sc, system, False, method=ox.BICGSTAB)
    assert s.resident_counts()[1] == 1
    for _ in range(40):
        _solve(sc, system, False)
    run = s.resident_counts()[0]
    for _ in range(80):
        _solve(sc, system, False, method=ox.BICGSTAB)
    assert s.resident_counts() == (run + 80, 1)
    s.close()


# (kind, shape, method, elimination): a thread per row, and the streamed matrix
SEVERAL = [("quad", (200, 199), ox.CG, ox.DIRICHLET_SYMMETRIC),
           ("quad", (150, 140), ox.BICGSTAB, ox.DIRICHLET_ROW),
           ("hex", (65, 64, 63), ox.CG, ox.DIRICHLET_SYMMETRIC),
           ("tet", (66, 64, 62), ox.BICGSTAB, ox.DIRICHLET_ROW)]


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("kind,shape,method,bc", SEVERAL)
def test_an_expired_wait_ends_the_solve(kind, shape, method, bc, prec):
    """Workgroups that take their first wait as run out (every one of them still
    runs to its end): the call fails, the solve is over and unconverged, and the next one
    finds nothing of it."""
    sc = _scenario(kind, shape)
    kw = dict(method=method, dirichlet=bc)
    system = W.make_system(sc, prec)
    s = system[1]
    ref = _solve(sc, system, True, **kw)
    s.resident_fail(ox.RESIDENT_EXPIRE)
    with pytest.raises(ox.OgsxError, match="too long"):
        _solve(sc, system, False, **kw)
    active, info = ox.solve_status(s)
    assert not active and info["converged"] == 0 and info["ret"] == 0
    run = s.resident_counts()[0]
    _same(_solve(sc, system, False, **kw), ref)
    assert s.resident_counts()[0] > run
    s.close()


def test_an_expired_wait_in_a_group():
    """The launch of the two quads expires: both are over, and the hexes, in a
    launch of their own, go on to the result they have alone.  Then the whole
    group again."""
    scs = [_scenario("quad", (90, 80)), _scenario("quad", (101, 70)), _scenario("hex", (22, 20, 18))]
    refs = []
    for sc in scs:
        system = W.make_system(sc, ox.FP64)
        refs.append(_solve(sc, system, True))
        system[1].close()
    systems = [W.make_system(sc, ox.FP64) for sc in scs]
    mem = [s for _, s in systems]
    g = ox.Group(ox.FP64)
    for s in mem:
        g.add(s)

    def start():
        for sc, s in zip(scs, mem):
            s.set_vector(ox.VEC_UOLD, sc.u0)
            s.set_vector(ox.VEC_X, sc.u0)
            s.initialize()
            s.assemble(sc.steps[0].dt, sc.steps[0].theta)
            s.set_dirichlet(sc.bc_idx, sc.bc_val, ox.DIRICHLET_SYMMETRIC)
        g.start(mem, method=ox.CG, tol=scs[0].tol, max_iter=40)

    def check(k):
        active, info = ox.solve_status(mem[k])
        assert not active
        _same((mem[k].get_vector(ox.VEC_X), info), refs[k])

    start()
    mem[0].resident_fail(ox.RESIDENT_EXPIRE)
    with pytest.raises(ox.OgsxError, match="too long"):
        g.advance(10)
    for s in mem[:2]:
        active, info = ox.solve_status(s)
        assert not active and info["converged"] == 0
    assert g.advance(1000) == 0
    check(2)
    start()
    assert g.advance(1000) == 0
    for k in range(3):
        check(k)
    g.close()
    for s in mem:
        s.close()


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("leaves", [1, 2, 3])
@pytest.mark.parametrize("kind,shape,method,bc", SEVERAL)
def test_solve_goes_on_where_a_launch_left(kind, shape, method, bc, leaves, prec):
    """Launches that leave (as when other work holds the chip): the solve goes on
    in separate launches, tries again, and after the third time no more; the
    iterates stay those of separate launches."""
    sc = _scenario(kind, shape)
    sc.max_iter = 3000
    kw = dict(method=method, dirichlet=bc)
    system = W.make_system(sc, prec)
    s = system[1]
    ref = _solve(sc, system, True, **kw)
    assert s.resident_counts() == (0, 0)
    s.resident_fail(ox.RESIDENT_LEAVE, leaves)
    _same(_solve(sc, system, False, **kw), ref)
    run, left = s.resident_counts()
    # (a solve of a few batches may end before its next try)
    assert 1 <= left <= leaves and (left < 3 or run == 0)
    s.resident_fail(ox.RESIDENT_LEAVE, 0)
    _same(_solve(sc, system, False, **kw), ref)
    assert s.resident_counts()[0] > run and s.resident_counts()[1] == left
    s.close()


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("kind,shape,method,bc", SEVERAL)
def test_resident_and_separate_launches_by_turns(kind, shape, method, bc, prec):
    """A launch that leaves between two that run, by small budgets of a group of
    one: resident, separate and resident iterations of one solve."""
    sc = _scenario(kind, shape)
    kw = dict(method=method, dirichlet=bc)
    system = W.make_system(sc, prec)
    ref = _solve(sc, system, True, **kw)
    s = system[1]
    s.set_vector(ox.VEC_UOLD, sc.u0)
    s.set_vector(ox.VEC_X, sc.u0)
    W._prepare_step(sc, s, 0, bc, False)
    g = ox.Group(prec)
    g.add(s)
    g.start([s], method=method, tol=sc.tol, max_iter=sc.max_iter)
    seen = []
    for budget, leave in ((5, 0), (7, 1), (3, 0), (6, 1)):
        before = s.resident_counts()
        s.resident_fail(ox.RESIDENT_LEAVE, leave)
        g.advance(budget)
        seen.append(tuple(b - a for a, b in zip(before, s.resident_counts())))
        if not ox.solve_status(s)[0]:
            break
    while g.advance(1000):
        pass
    # run; left; separate (the wait after a leave); run again or left
    assert seen[0] == (1, 0) and (0, 1) in seen
    _same((s.get_vector(ox.VEC_X), ox.solve_status(s)[1]), ref)
    g.close()
    s.close()


def _star(leaves):
    """Line elements from one node: its row has leaves + 1 entries."""
    from ogs5_amd.mesh import LINE2, Mesh
    z = np.zeros(leaves + 1)
    x = np.concatenate([[0.0], 1.0 + np.arange(leaves) / leaves])
    conn = np.stack([np.zeros(leaves, np.int64), np.arange(1, leaves + 1)], 1)
    sc = _scenario("line", (leaves,))
    sc.mesh = Mesh(LINE2, 1, x, z, z.copy(), conn, (leaves,), (1.0,), np.arange(leaves))
    sc.bc_idx, sc.bc_val = np.array([0]), np.array([1.0])
    return sc


# longest rows and most rows of each kind of launch, and one past them
@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("make,method,fits", [
    (lambda: _star(26), ox.CG, True), (lambda: _star(27), ox.CG, False),
    # (past 27 entries BiCGStab streams a matrix with a stencil dictionary)
    (lambda: _star(26), ox.BICGSTAB, True), (lambda: _star(27), ox.BICGSTAB, True),
    (lambda: _scenario("quad", (511, 511), permute=True), ox.CG, True),
    (lambda: _scenario("quad", (512, 511), permute=True), ox.CG, False),
    (lambda: _scenario("quad", (512, 511)), ox.CG, True),
    (lambda: _scenario("quad", (361, 361), permute=True), ox.BICGSTAB, True),
    (lambda: _scenario("quad", (361, 362), permute=True), ox.BICGSTAB, False),
    (lambda: _scenario("quad", (361, 362)), ox.BICGSTAB, True)])
def test_sizes_that_run_resident(make, method, fits, prec):
    """... and profiling, which keeps a solve to separate launches."""
    sc = make()
    sc.max_iter = 12
    kw = dict(method=method, dirichlet=ox.DIRICHLET_ROW if method == ox.BICGSTAB
              else ox.DIRICHLET_SYMMETRIC)
    system = W.make_system(sc, prec)
    s = system[1]
    ref = _solve(sc, system, True, **kw)
    assert s.resident_counts() == (0, 0)
    _same(_solve(sc, system, False, **kw), ref)
    assert (s.resident_counts()[0] > 0) == fits and s.resident_counts()[1] == 0
    s.close()


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
@pytest.mark.parametrize("method,bc", [(ox.CG, ox.DIRICHLET_SYMMETRIC), (ox.BICGSTAB, ox.DIRICHLET_ROW)])
@pytest.mark.parametrize("fmt,joins", [(5, True), (9, True), (0, False)])
def test_small_members_join_separate_launches(method, bc, prec, fmt, joins):
    """A group where one member has a format set, and so separate launches: the
    small others go along in them, in its format, and take resident ones once it
    is done; where none does, all are resident."""
    scs = [_scenario("quad", (31, 30), seed=1), _scenario("quad", (40, 33), permute=True),
           _scenario("quad", (52, 47), permute=True)]
    refs, mem = [], []
    for sc in scs:
        sc.max_iter = 30
        system = W.make_system(sc, prec)
        refs.append(_solve(sc, system, True, method=method, dirichlet=bc))
        system[1].close()
        mem.append(W.make_system(sc, prec)[1])
    mem[0].set_spmv_variant(fmt)
    g = ox.Group(prec)
    for s in mem:
        g.add(s)
    for sc, s in zip(scs, mem):
        s.set_vector(ox.VEC_UOLD, sc.u0)
        s.set_vector(ox.VEC_X, sc.u0)
        W._prepare_step(sc, s, 0, bc, False)
    g.start(mem, method=method, tol=scs[0].tol, max_iter=30)
    g.advance(3)
    assert [s.resident_counts()[0] > 0 for s in mem[1:]] == [not joins] * 2
    if fmt:
        assert [s.spmv_format(fp32=prec == ox.FP32_IR) for s in mem[1:]] == [fmt] * 2
    while g.advance(1000):
        pass
    for k in (1, 2):
        active, info = ox.solve_status(mem[k])
        _same((mem[k].get_vector(ox.VEC_X), info), refs[k])
    g.close()
    for s in mem:
        s.close()


@pytest.mark.parametrize("kind,shape,method,bc,prec,max_iter", [
    # FP64 with x in memory (3 vectors in LDS), and with p there too
    ("hex", (105, 105, 105), ox.CG, ox.DIRICHLET_SYMMETRIC, ox.FP64, 1500),
    ("hex", (120, 120, 118), ox.CG, ox.DIRICHLET_SYMMETRIC, ox.FP64, 1000),
    ("quad", (200, 199), ox.BICGSTAB, ox.DIRICHLET_ROW, ox.FP64, 4500),
    ("tet", (80, 72, 64), ox.BICGSTAB, ox.DIRICHLET_ROW, ox.FP64, 1500)])
def test_a_launch_holds_the_chip_for_a_bounded_time(kind, shape, method, bc, prec, max_iter):
    """No launch takes much more than 10 ms, whatever its system: its iterations
    go by what one of them costs.  (A tolerance that no solve reaches.)"""
    sc = _scenario(kind, shape)
    kw = dict(method=method, dirichlet=bc)
    system = W.make_system(sc, prec)
    s = system[1]
    ref = _solve(sc, system, True, **kw)
    _same(_solve(sc, system, False, **kw), ref)
    W._prepare_step(sc, s, 0, bc, False)
    before = s.resident_counts()[0]
    t = time.perf_counter()
    info = s.solve(method=method, tol=1e-300, max_iter=max_iter)
    t = time.perf_counter() - t
    run = s.resident_counts()[0] - before
    print(f"{info['iterations']} iterations, {run} launches, {1e3 * t:.1f} ms")
    assert run > 1 and t / run < 0.02
    s.close()


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
def test_solves_leave_the_tuned_format(prec):
    """A streamed BiCGStab solve reads the matrix through the stencil dictionary,
    whatever the tuner found; after it, and where profiling keeps it to separate
    launches, the tuner's format is in use."""
    sc = _scenario("hex", (65, 64, 63))
    kw = dict(method=ox.BICGSTAB, dirichlet=ox.DIRICHLET_ROW)
    system = W.make_system(sc, prec)
    s = system[1]

    def formats():
        return s.spmv_format(), s.spmv_format(fp32=True)

    ref = _solve(sc, system, True, **kw)
    tuned = formats()
    print(f"tuned formats {tuned}")
    _same(_solve(sc, system, False, **kw), ref)
    assert s.resident_counts()[0] > 0
    assert formats() == tuned
    _same(_solve(sc, system, True, **kw), ref)
    assert formats() == tuned
    s.close()


@pytest.mark.parametrize("prec", [ox.FP64, ox.FP32_IR])
def test_solves_at_once(prec):
    """Three solves on their own streams, from threads of their own: a streamed
    one that takes every compute unit and two of a thread per row, whose launches
    find the chip taken now and then.  Each gives its own bits every time."""
    import threading
    scs = [_scenario("hex", (70, 68, 66)), _scenario("quad", (200, 199)), _scenario("quad", (300, 290))]
    for sc in scs:
        sc.max_iter = 120
    refs, systems = [], []
    for sc in scs:
        systems.append(W.make_system(sc, prec))
        refs.append(_solve(sc, systems[-1], True))
        systems[-1][1].profile(False)
    got = [[] for _ in scs]

    def work(k):
        for _ in range(8):
            got[k].append(_solve(scs[k], systems[k], False))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print([s.resident_counts() for _, s in systems])
    for k in range(3):
        assert len(got[k]) == 8 and systems[k][1].resident_counts()[0] > 0
        for r in got[k]:
            _same(r, refs[k])
        systems[k][1].close()
